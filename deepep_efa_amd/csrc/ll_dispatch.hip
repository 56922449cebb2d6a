// Low-latency dispatch: route ranking, fused quantise + pack (send side),
// segment compaction (receive side), and the single launch that runs both
// for decode-sized batches.
//
// Data layout in HBM (row stride S = row_stride_bytes(H, format)):
//   recv_staging  [E_l][R][M] rows — slot j of segment (e_l, s) is the j-th
//                 row rank s sent to local expert e_l, in ascending (t,k)
//                 order of the sender.
//   recv_count    [E_l][R] int32 — rows present in each segment.
//   send_slots    [E][M] rows — this rank's rows for remote experts.
// A staged row is [data | pad16][scales | pad16][src_token, k, src_rank, local expert].
//
// Work is cut per wavefront, never per thread block: one wave owns one 1 KiB
// piece of one row, so a 64-lane 16-byte access is one contiguous KiB and no
// LDS or barrier is needed on the copy paths.
#include "common.hpp"
#include "quant.hpp"
#include "segments.hpp"
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "../../include/deepep_hip.h"

// Route scratch (the chunk histograms of ll_rank_chunk_kernel) for deepep_ll_dispatch_send_static,
// whose callers cannot allocate.  The array is part of the code object: every GPU the library runs
// on holds its own copy, at its own address, until the process ends.  Host code never passes this
// name to a kernel; it passes the device address hipGetSymbolAddress returns (static_route_scratch).
constexpr size_t kStaticScratchBytes = size_t(1) << 20;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];

namespace deepep {

__host__ __device__ inline int64_t align256(int64_t v) { return (v + 255) & ~int64_t(255); }

constexpr int kRankChunkEntries = 2048;  // entries of a chunk, at most
constexpr int kSendColumns = 32;         // chunks whose histograms the waves that store the rows add up themselves
// The send kernel ranks its own slots up to here, which costs its rows less than a launch ahead of them costs the stream.
constexpr int kSelfRankMaxEntries = 8192;

// Tokens of a chunk: whole ones, about kRankChunkEntries entries.
inline int rank_chunk_tokens(int num_topk) {
    const int t = kRankChunkEntries / num_topk;
    return t < 1 ? 1 : t;
}

// The chunk histograms, int32 [chunks][E].
static int64_t chunk_hist_bytes(int num_tokens, int num_topk, int num_experts) {
    const int tpc = rank_chunk_tokens(num_topk);
    const int64_t chunks = (num_tokens + tpc - 1) / tpc;
    return align256((chunks < 1 ? 1 : chunks) * num_experts * 4);
}
// Per source: the chunk histograms, where an own expert's rows begin, int32 [E], and slots, int32 [T][K].
static int64_t route_scratch_bytes(int num_tokens, int num_topk, int num_experts) {
    return chunk_hist_bytes(num_tokens, num_topk, num_experts) + align256(int64_t(num_experts) * 4) +
           align256(int64_t(num_tokens) * num_topk * 4);
}

// Entries that name expert e in the first num_chunks chunk histograms.
__device__ __forceinline__ int chunk_total(const int32_t* __restrict__ hists, int num_chunks, int num_experts, int e) {
    int total = 0;
    for (int c0 = 0; c0 < num_chunks; c0 += 8) {  // eight loads in flight
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = c0 + u < num_chunks ? hists[int64_t(c0 + u) * num_experts + e] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) total += v[u];
    }
    return total;
}

// Writes the per-expert totals where the receivers look for them.
__device__ __forceinline__ void emit_expert_count(int e, int total, int num_experts, int num_ranks, int rank,
                                                  int src_rank, int max_tokens, int32_t* recv_count,
                                                  int32_t* send_count) {
    const int cnt = total < max_tokens ? total : max_tokens;
    const int experts_per_rank = num_experts / num_ranks;
    if (send_count != nullptr) send_count[e] = cnt;
    if (e / experts_per_rank == rank) recv_count[(e % experts_per_rank) * num_ranks + src_rank] = cnt;
}

// ---------------------------------------------------------------------
// Fused quantise + pack.  A workgroup owns one token (of one source); each of
// its waves owns one (1 KiB output piece, share of the K selections).
// FP8 formats: the piece is 8 scale groups (1024 channels, 2 KiB of bf16 in);
// each 8-lane cluster owns a group, each lane 16 channels.  The quantised
// 16 bytes stay in registers and are stored once per selection — the row is
// read and quantised once however many experts it goes to
// (reference idea: csrc/kernels/coop_dispatch_send.cuh:572-607).
//
// Per-selection bookkeeping (slot, destination row address, row tail,
// pair_slot) is done once per workgroup by the first lanes of wave 0, one for
// each selection of its one, two or four tokens (at most 64), and handed to the
// other waves through LDS; each wave reads its token's K destinations with one
// LDS access and takes them back per selection with readlane.  Quantisation runs
// while wave 0 does that.  Barriers fence LDS only, so the row loads stay in
// flight across them.
//
// The slot of a selection is the number of earlier (token,k) entries naming its
// expert (reference: the serial scan of csrc/kernels/efa_kernels.cu:617-637 and
// token_offset / expert_offsets of csrc/kernels/coop_dispatch_send.cuh:360-420).
// Up to kSelfRankMaxEntries entries, and in the single-launch dispatch for as many
// as dispatch_in_one_launch() lets it have, the workgroup counts them itself: while
// the row loads are in flight every thread fetches up to four entries that precede
// the token (more in a loop) and adds them to a histogram by expert in LDS; the
// per-expert totals come from one extra workgroup per source.  Larger batches get
// their slots from ll_rank_chunk_kernel, one launch ahead.  Deterministic: integer
// adds only.
// ---------------------------------------------------------------------
constexpr int kMaxTopk = 64;
constexpr int kFusedMaxEntries = 8192;     // send + receive in one launch up to here, whatever the rows
constexpr int kSendMaxWaves = 16;

// A workgroup that ranks its own slots takes two or four tokens where it has waves for them, and one sweep through the
// entries serves them all: while that leaves 240 workgroups of them, about one for every compute unit.  The sweeps are
// instructions and LDS adds on every compute unit; so are the receive workgroups' for the own counts in the single-launch
// dispatch, of which there are half as many then, 512 instead of 1024 (640 give 0.7 us of the first figure back).  There
// it pays where a row has one or two pieces and four waves are more than a token takes.  Microseconds of a step or an
// exchange, one token a workgroup / several:
//   step, 1000 x 2048     39.2 / 36.3     exchange, 1000 x 2048  47.2 / 44.8     step, 509 x 4096  23.5 / 23.8 and 24.4 / 23.9
//   700 x 2048            28.6 / 27.4     700 x 2048             38.4 / 36.8     400 x 4096, in 200 workgroups  28.6 / 30.2
//   900 x 2048, top-6     31.2 / 29.7     1000 x 5120            91.1 / 87.6     700 x 4096        42.0 / 41.7
//   500 x 2048            22.2 / 21.4                                            1000 x 4096       57.5 / 57.4
// A send of its own fits two tokens in up to sixteen waves.  In more than eight of them it pays from 480 workgroups and 4096
// entries on, in twelve, and in sixteen by destination, whose tokens go through all entries; fourteen leave four of a compute
// unit's places empty.  Microseconds of the send alone, one token a workgroup / two, staged and by destination:
//   960 x 3072     9.7 /  9.3  10.7 /  9.4     1000 x 4096  10.8 / 10.8  12.3 / 11.1     1000 x 7168        14.8 / 14.3  15.8 / 15.4
//   1000 x 5120   11.8 / 11.6  14.4 / 13.0     600 x 4096    8.3 /  9.1   8.7 / 10.1     2000 x 7168, top-4 16.5 / 19.0  18.8 / 20.3
//   600 x 3072     7.7 /  8.0   8.2 /  8.0     1500 x 5120, top-2  8.6 / 9.1  10.0 / 9.9    600 x 7168       10.0 / 11.6  11.2 / 11.7
constexpr int kManyBlocks = 240;
constexpr int kTwoTokensFrom = 4096;  // entries

struct ByDestTables {
    int32_t* expert_prefix;  // [E + 1]
    int32_t* rank_counts;    // [R]
    int64_t* rank_cumsum;    // [R + 1]
};

struct SendArgs {
    const uint8_t* x;
    const int64_t* topk_idx;
    const int32_t* src_ranks;  // null: the rows are this rank's own
    int num_tokens, hidden, num_topk, num_experts, num_ranks, rank, max_tokens;
    int pieces_per_row, split_log2;
    int tokens_per_block;  // 1, 2 or 4: whole tokens, pieces_per_row << split_log2 waves each
    RankDivider token_of;  // a workgroup's entry to the token among its own: division by K
    uint32_t rank_of_expert_magic;
    uint8_t* recv_staging;
    uint8_t* send_slots;
    int32_t* pair_slot;
    int32_t* recv_count;
    int32_t* send_count;
    // By-destination form: send_slots is one buffer of rows, contiguous per destination rank, and every
    // row (the rank's own included) goes to row expert_prefix[expert] + slot of it.  Null: per-expert slots.
    const int32_t* expert_prefix;
    // By-destination batches that rank themselves: every token's workgroup gets the batch's entries per
    // expert itself, and the counting row writes the tables out.
    int prefix_in_block;
    ByDestTables by_dest;
};

// A batch ranked ahead of its rows, a chunk of tokens at a time.
struct RankedBatch {
    int num_chunks, tokens_per_chunk;
    RankDivider chunk_of;       // a token's chunk
    const int32_t* hists;       // [chunks][E] entries of a chunk that name an expert
    int32_t* slots;             // [T][K] slots, counted within the chunk or, in_full, within the batch
    int64_t stride;             // of both from a source to the next, in ints
    int in_full;
    int32_t* own_first;         // [E_l] where the rank's own rows begin (null: nobody asks)
    int first_in_finish;        // the launch between the two writes own_first, over the last chunk's histogram
};

// Final destination of the rows a rank sends to its own experts, used by the
// one-call dispatch (as one launch or two): they skip the staging area and land
// in the packed tensors behind the rows of the lower source ranks, which is where
// the reference's ascending-source ranges put them.
struct DirectOut {
    uint8_t* packed_x;  // null: stage own rows like everyone else's
    uint8_t* packed_scales;
    int32_t* src_info;
};

// Top-k entries read two at a time, with zeros past the end of the list: 16-byte loads, which as buffer loads need no
// more than the four-byte alignment that every list has.
struct EntryPair {
    u32x4 v;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t list, int pair) { v = load_row_u32x4<false>(list, pair * 16); }
    // Entry 0 or 1 as an expert below `limit` counted from `first`, if it names one.
    __device__ __forceinline__ bool expert(int which, uint32_t first, uint32_t limit, uint32_t& e) const {
        e = v[which * 2] - first;
        return (v[which * 2 + 1] == 0u) & (e < limit);
    }
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t entry_list(const int64_t* topk_idx, int n) {
    return row_buffer(reinterpret_cast<const uint8_t*>(topk_idx), n * 8);
}

struct alignas(16) SendLds {
    uint64_t sel_row[kMaxTopk];    // where selection k's payload goes (0: nowhere)
    uint64_t sel_scale[kMaxTopk];  // where its scales go
};

// hist[e] (LDS, [E + 1]) = entries of topk_idx[0 .. n) naming expert e, clamped to max_tokens, then their
// exclusive prefix over the experts with the total in hist[E]; the whole workgroup takes part.
// counts_out: the clamped counts.
__device__ __forceinline__ void expert_prefix_in_lds(const int64_t* __restrict__ topk_idx, int n, int num_experts,
                                                     int max_tokens, int32_t* hist, int32_t* wave_totals,
                                                     int32_t* counts_out) {
    const int tid = threadIdx.x, threads = block_threads();
    for (int e = tid; e < num_experts; e += threads) hist[e] = 0;
    lds_barrier();
    constexpr int kAhead = 4;  // pairs of entries in flight per thread
    const auto list = entry_list(topk_idx, n);
    for (int base = tid; base * 2 < n; base += kAhead * threads) {
        EntryPair ahead[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) ahead[u].load(list, base + u * threads);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                uint32_t e;
                if (ahead[u].expert(i, 0, uint32_t(num_experts), e) && (base + u * threads) * 2 + i < n)
                    atomicAdd(&hist[e], 1);
            }
    }
    lds_barrier();
    for (int e = tid; e < num_experts; e += threads) {
        const int c = hist[e] < max_tokens ? hist[e] : max_tokens;
        hist[e] = c;
        counts_out[e] = c;
    }
    lds_barrier();
    block_exclusive_scan(hist, num_experts, wave_totals);
}

// For one wave: the rows of the experts before the lane's expert e (none: e < 0), an expert's entries -- the low half
// of its word of hist (LDS) -- clamped to max_tokens.  Lane l adds up the l-th 64th of the experts.
__device__ __forceinline__ int wave_expert_prefix(const int32_t* hist, int num_experts, int max_tokens, int e) {
    const int per = (num_experts + kWave - 1) / kWave, lane = lane_id();
    const auto rows_of = [&](int x) {
        const int c = hist[x] & 0xffff;
        return c < max_tokens ? c : max_tokens;
    };
    int sum = 0;
    for (int j = 0; j < per; ++j)
        if (lane * per + j < num_experts) sum += rows_of(lane * per + j);
    const int base = wave_inclusive_sum(sum) - sum;
    const int owner = e < 0 ? 0 : e / per;
    int run = __shfl(base, owner, kWave);
    for (int j = 0; j < per; ++j)
        if (owner * per + j < e) run += rows_of(owner * per + j);
    return run;
}

// The per-rank tables of the by-destination form from the prefix in LDS.
__device__ __forceinline__ void by_dest_tables_out(const int32_t* hist, int num_experts, int num_ranks,
                                                   const ByDestTables& out) {
    const int tid = threadIdx.x, threads = block_threads();
    for (int e = tid; e <= num_experts; e += threads) out.expert_prefix[e] = hist[e];
    const int experts_per_rank = num_experts / num_ranks;
    for (int r = tid; r < num_ranks; r += threads) {
        out.rank_counts[r] = hist[(r + 1) * experts_per_rank] - hist[r * experts_per_rank];
        out.rank_cumsum[r] = hist[r * experts_per_rank];
    }
    if (tid == 0) out.rank_cumsum[num_ranks] = hist[num_experts];
}

// The per-source counting workgroup.
__device__ __forceinline__ void send_count_block(const SendArgs& a, int b, int32_t* lds_hist) {
    const int tid = threadIdx.x;
    const int n = a.num_tokens * a.num_topk;
    const int src_rank = a.src_ranks != nullptr ? a.src_ranks[b] : a.rank;
    const int64_t* my_topk = a.topk_idx + int64_t(b) * n;
    for (int j = tid; j < a.num_experts; j += block_threads()) lds_hist[j] = 0;
    lds_barrier();
    for (int i = tid; i < n; i += block_threads()) {
        const int64_t v = my_topk[i];
        if (v >= 0 && v < a.num_experts) atomicAdd(&lds_hist[int(v)], 1);
    }
    lds_barrier();
    for (int e = tid; e < a.num_experts; e += block_threads())
        emit_expert_count(e, lds_hist[e], a.num_experts, a.num_ranks, a.rank, src_rank, a.max_tokens, a.recv_count,
                          a.send_count);
}

// A wave's stores of its piece, one a selection of its part: lane k holds selection k's row and scales (0: nowhere), which
// the loop takes back as wave-uniform values.
template <int kFmt, bool kStream>
__device__ __forceinline__ void store_selections(uint64_t my_row, uint64_t my_scale_row, int num_topk, int part, int split,
                                                 int data_bytes, int scale_bytes, int lane_off, u32x4 payload,
                                                 int scale_off, uint32_t scale_bits) {
    for (int k = part; k < num_topk; k += split) {
        const uint8_t* row = reinterpret_cast<const uint8_t*>(
            (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(my_row >> 32), k))) << 32) |
            uint32_t(__builtin_amdgcn_readlane(int(uint32_t(my_row)), k)));
        if (row == nullptr) continue;
        store_row_u32x4<kStream>(row_buffer(row, data_bytes), lane_off, payload);
        if constexpr (kFmt != kRowBF16) {
            const uint8_t* scale_row = reinterpret_cast<const uint8_t*>(
                (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(my_scale_row >> 32), k))) << 32) |
                uint32_t(__builtin_amdgcn_readlane(int(uint32_t(my_scale_row)), k)));
            const auto scales = row_buffer(scale_row, scale_bytes);
            if constexpr (kFmt == kRowFP8UE8M0)
                __builtin_amdgcn_raw_buffer_store_b8(uint8_t(scale_bits >> 23), scales, scale_off, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b32(scale_bits, scales, scale_off, 0, 0);
        }
    }
}

// One workgroup's share of token t of source b.  kStream (64 MB of traffic and more): the payload of
// the rows is stored with the non-temporal hint; at 4096 tokens, with the
// destinations in HBM, that takes the send from 73 to 53 us (a row stored the ordinary way is first
// allocated in the memory-side cache and written back later).  The token rows are read, and the
// scales and tails stored, the ordinary way: the hint measured slower on those (63 and 56 us).
// kTables: the launch may be one that makes the by-destination tables.
// kMany: the workgroup's share are the tokens_per_block tokens from t on, which are ranked by one sweep; lane i of wave 0
// has the i-th of their selections.
template <int kFmt, bool kStream, bool kTables, bool kMany>
__device__ __forceinline__ void send_token_block(const SendArgs& a, const DirectOut& direct, int b, int t,
                                                 int block_in_token, SendLds& lds, int32_t* lds_hist) {
    const int lane = lane_id(), tid = threadIdx.x;
    const int num_topk = a.num_topk, num_experts = a.num_experts;
    const int waves_per_token = a.pieces_per_row << a.split_log2;
    const int n = a.num_tokens * num_topk;
    const int src_rank = a.src_ranks != nullptr ? a.src_ranks[b] : a.rank;
    const int64_t* my_topk = a.topk_idx + int64_t(b) * n;

    int item = block_in_token * (block_threads() >> 6) + wave_in_block(), token = 0;  // of the workgroup's, this wave's
    if constexpr (kMany)
        while (item >= waves_per_token && token + 1 < a.tokens_per_block) item -= waves_per_token, ++token;
    const int split = 1 << a.split_log2;
    const bool wave_live = item < waves_per_token && t + token < a.num_tokens;
    const int part = item & (split - 1);
    const int piece = item >> a.split_log2;
    const int64_t row_id = int64_t(b) * a.num_tokens + (wave_live ? t + token : t);
    const int entry0 = t * num_topk;
    const int selections = kMany ? min(a.tokens_per_block * num_topk, n - entry0) : num_topk;

    const int64_t data_bytes = row_data_bytes(a.hidden, kFmt);
    const int64_t data_pad = align16(data_bytes);
    const int64_t scale_bytes = row_scale_bytes(a.hidden, kFmt);
    const int64_t scale_pad = align16(scale_bytes);
    const int64_t stride = row_stride_bytes(a.hidden, kFmt);

    DEEPEP_PHASE(0);
    // ---- issue this wave's row loads ------------------------------------
    const auto token_row = row_buffer(a.x + uint64_t(row_id) * (uint32_t(a.hidden) * 2), a.hidden * 2);
    u32x4 lo, hi = {0u, 0u, 0u, 0u};  // zeros past the row's end
    bool lane_live = wave_live;
    int group = 0;
    if constexpr (kFmt == kRowBF16) {
        lo = load_row_u32x4<false>(token_row, piece * 1024 + lane * 16);
    } else {
        group = piece * 8 + (lane >> 3);
        lane_live = wave_live && group < a.hidden / kGroup;
        lo = load_row_u32x4<false>(token_row, piece * 2048 + lane * 32);
        hi = load_row_u32x4<false>(token_row, piece * 2048 + lane * 32 + 16);
    }

    // ---- every index load of the ranking, issued before anything waits -----
    // The loads are unconditional (an index that is not wanted is clamped to one that exists and its
    // value dropped): without branches around them the compiler can count them, so the first wait of
    // wave 0 -- for the token's own selections -- does not also wait out a second round trip for the
    // entries it sweeps.
    const int threads = block_threads();
    const bool prefix_in_block = kTables && a.prefix_in_block;
    const int sweep_end = prefix_in_block ? n : entry0;
    constexpr int kSweepAhead = 2;
    const int64_t own_v = my_topk[entry0 + (tid < selections ? tid : selections - 1)];  // thread i: selection i
    const auto list = entry_list(my_topk, n);
    const int sweep_pairs = (sweep_end + 1) >> 1;
    EntryPair ahead[kSweepAhead];
#pragma unroll
    for (int r = 0; r < kSweepAhead; ++r) ahead[r].load(list, tid + r * threads);
    for (int e = tid; e < num_experts; e += threads) lds_hist[e] = 0;
    lds_barrier();

    // ---- per-selection bookkeeping, once per token --------------------------
    int my_expert = -1, my_slot = -1, dst_rank = -1, local = 0;  // thread i: selection i
    int direct_begin = 0;
    if (tid < selections) {
        const int64_t v = own_v;
        if (v >= 0 && v < num_experts) {
            my_expert = int(v);
            // my_expert / E_l by multiply-high; magic 0 stands for E_l == 1
            dst_rank = a.rank_of_expert_magic != 0 ? int(__umulhi(uint32_t(my_expert), a.rank_of_expert_magic))
                                                   : my_expert;
            local = my_expert - dst_rank * (num_experts / a.num_ranks);
        }
    }
    int dest_first = 0;  // by-destination form: where the expert's run of rows begins in the send buffer
    if (direct.packed_x != nullptr && tid < kWave) {
        // Rows for this rank's own experts go straight to the packed tensors, at the place the
        // reference's range builder gives them: behind the rows of the lower source ranks
        // (csrc/kernels/efa_kernels.cu:991-1010).  For each such selection wave 0 adds up those
        // ranks' counts of the expert, kOwn of them at a time where there are several tokens'.
        constexpr int kOwn = kMany ? 4 : 1;
        uint64_t to_own = __ballot(my_expert >= 0 && dst_rank == a.rank);
        while (to_own != 0) {
            int k[kOwn], counts_at[kOwn], part[kOwn];
#pragma unroll
            for (int u = 0; u < kOwn; ++u) {
                k[u] = to_own != 0 ? __builtin_ctzll(to_own) : (u > 0 ? k[u - 1] : 0);  // again the one before
                to_own &= to_own - 1;
                counts_at[u] = __builtin_amdgcn_readlane(local, k[u]) * a.num_ranks;
                part[u] = 0;
            }
            for (int s = lane; s < a.rank; s += kWave) {
                int c[kOwn];
#pragma unroll
                for (int u = 0; u < kOwn; ++u) c[u] = a.recv_count[counts_at[u] + s];
#pragma unroll
                for (int u = 0; u < kOwn; ++u) part[u] += c[u] < 0 ? 0 : (c[u] > a.max_tokens ? a.max_tokens : c[u]);
            }
#pragma unroll
            for (int u = 0; u < kOwn; ++u) {
                const int sum = __builtin_amdgcn_readlane(wave_inclusive_sum(part[u]), kWave - 1);
                if (lane == k[u]) direct_begin = sum;
            }
        }
    }
    DEEPEP_PHASE(1);
    u32x4 payload = lo;  // quantised below, while the workgroup's bookkeeping is in flight
    uint32_t scale_bits = 0;
    // Rank the selections: the entries between the start of the sweep and this token, counted by expert in LDS.  (A
    // ballot for each selection and load instead cost every wave of the workgroup 130 instructions a round of four
    // entries a thread: 128 tokens 7.7 -> 7.4 us, 300 tokens 15.9 -> 15.4, single entries read instead of pairs 16.1.)
    // With prefix_in_block the sweep goes through the whole batch: the low half of a word counts all of its entries and
    // the high half those before the token, and wave 0 gets the prefix from the same words (128 tokens 9.4 -> 7.8 us
    // against a histogram of its own and a scan by the whole workgroup).
    const int before = prefix_in_block ? 0x10001 : 1;
    const auto count_pair = [&](int pair, const EntryPair& entries) {
        if (pair >= sweep_pairs) return;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int at = pair * 2 + i;
            uint32_t e;
            if (entries.expert(i, 0, uint32_t(num_experts), e) && at < sweep_end)
                atomicAdd(&lds_hist[e], at < entry0 ? before : 1);
        }
    };
#pragma unroll
    for (int r = 0; r < kSweepAhead; ++r) count_pair(tid + r * threads, ahead[r]);
    for (int base = kSweepAhead * threads; base < sweep_pairs; base += kSweepAhead * threads) {
#pragma unroll
        for (int r = 0; r < kSweepAhead; ++r) ahead[r].load(list, base + tid + r * threads);
#pragma unroll
        for (int r = 0; r < kSweepAhead; ++r) count_pair(base + tid + r * threads, ahead[r]);
    }
    if constexpr (kFmt != kRowBF16) payload = quantise_16<kFmt>(lo, hi, scale_bits);
    lds_barrier();
    DEEPEP_PHASE(3);
    if (tid < kWave) {  // wave 0: lane k finishes selection k
        int total = my_expert >= 0 ? lds_hist[my_expert] : 0;
        if (prefix_in_block) {
            total = int(uint32_t(total) >> 16);
            dest_first = wave_expert_prefix(lds_hist, num_experts, a.max_tokens, my_expert);
        }
        if constexpr (kMany) {  // the same expert named earlier in these tokens
            uint64_t same = __ballot(my_expert >= 0);
            for (int bit = 1; bit < num_experts; bit <<= 1) {
                const uint64_t votes = __ballot((my_expert & bit) != 0);
                same &= (my_expert & bit) != 0 ? votes : ~votes;
            }
            total += __popcll(same & lanes_below(lane));
        } else {
            for (int k2 = 0; k2 < num_topk; ++k2) {  // the same expert named earlier in this token
                const int other = __builtin_amdgcn_readlane(my_expert, k2);
                if (k2 < tid && other == my_expert) total += 1;
            }
        }
        if (tid < selections && my_expert >= 0) my_slot = total;
    }
    if (tid < selections) {
        const int of_token = kMany ? a.token_of(tid) : 0;
        if (my_slot >= a.max_tokens) my_slot = -1;
        uint8_t* row = nullptr;
        uint8_t* scale_row = nullptr;
        bool staged = false;
        if (my_slot >= 0) {
            if (a.expert_prefix != nullptr) {
                row = a.send_slots + (int64_t(dest_first) + my_slot) * stride;
                staged = true;
            } else if (dst_rank == a.rank && direct.packed_x != nullptr) {
                const int64_t out_row = int64_t(local) * a.num_ranks * a.max_tokens + direct_begin + my_slot;
                row = direct.packed_x + out_row * data_bytes;
                scale_row = direct.packed_scales + out_row * scale_bytes;
                if (block_in_token == 0) direct.src_info[out_row] = t + of_token;
            } else if (dst_rank == a.rank) {
                row = a.recv_staging + ((int64_t(local) * a.num_ranks + src_rank) * a.max_tokens + my_slot) * stride;
                staged = true;
            } else if (a.send_slots != nullptr) {
                row = a.send_slots + (int64_t(my_expert) * a.max_tokens + my_slot) * stride;
                staged = true;
            }
            if (staged) scale_row = row + data_pad;
        }
        lds.sel_row[tid] = reinterpret_cast<uint64_t>(row);
        lds.sel_scale[tid] = reinterpret_cast<uint64_t>(scale_row);
        if (block_in_token == 0) {
            if (a.pair_slot != nullptr) a.pair_slot[entry0 + tid] = my_slot;
            if (staged) {
                u32x4 tail = {uint32_t(t + of_token), uint32_t(tid - of_token * num_topk), uint32_t(src_rank), uint32_t(local)};
                *reinterpret_cast<u32x4*>(row + data_pad + scale_pad) = tail;
            }
        }
    }
    lds_barrier();
    DEEPEP_PHASE(4);
    if (!wave_live) return;

    // ---- one store per selection ----------------------------------------
    // Rows are addressed as buffers: lanes past a row's end and, with the scales, all but the first of eight store
    // nothing without a mask of their own.
    const int lane_off = piece * 1024 + lane * 16;
    const int scale_off = lane_live && (lane & 7) == 0 ? (kFmt == kRowFP8UE8M0 ? group : group * 4) : 0x7fffffff;
    DEEPEP_PHASE(5);
    // lane k reads selection k's destinations once
    uint64_t my_row = 0, my_scale_row = 0;
    if (lane < num_topk) {
        my_row = lds.sel_row[token * num_topk + lane];
        my_scale_row = lds.sel_scale[token * num_topk + lane];
    }
    store_selections<kFmt, kStream>(my_row, my_scale_row, num_topk, part, split, int(data_bytes), int(scale_bytes), lane_off,
                                    payload, scale_off, scale_bits);
    DEEPEP_PHASE(6);
}

template <int kFmt, bool kStream, bool kMany>
__global__ __launch_bounds__(kSendMaxWaves* kWave) void ll_send_kernel(SendArgs a) {
    extern __shared__ int32_t lds_hist[];  // [E + 1]
    __shared__ SendLds lds;
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    if (blockIdx.y + 1 == gridDim.y) {  // the counting row of the grid
        if (blockIdx.x != 0) return;
        if (a.prefix_in_block) {  // this workgroup writes the tables out
            expert_prefix_in_lds(a.topk_idx, a.num_tokens * a.num_topk, a.num_experts, a.max_tokens, lds_hist, wave_totals,
                                 a.send_count);
            by_dest_tables_out(lds_hist, a.num_experts, a.num_ranks, a.by_dest);
        } else {
            send_count_block(a, blockIdx.z, lds_hist);
        }
        return;
    }
    send_token_block<kFmt, kStream, true, kMany>(a, DirectOut{nullptr, nullptr, nullptr}, blockIdx.z,
                                                 int(blockIdx.y) * (kMany ? a.tokens_per_block : 1), blockIdx.x, lds, lds_hist);
}

// ---------------------------------------------------------------------
// Large batches: the entries are ranked one launch ahead of the rows, four workgroups a chunk, 512 entries each.  A wave
// matches its 64 entries against one another, a ballot for each bit of the expert, and leaves how many it has of an expert
// in a byte of LDS; an entry's place in its chunk is what the parts before its own hold of its expert, counted by LDS adds,
// what the waves before its own do, and the lanes before it.  The last part has all it takes for the chunk's histogram,
// and what the chunks before an entry's hold of its expert is added by whoever reads the place.  Latency and instructions
// bound it: four SIMDs issue for the whole of a workgroup.  One workgroup a chunk, two entries a lane, took a microsecond
// longer: both launches of a send by destination of 2047 tokens of 7168 30.5 us against 29.5, of 1100 20.2 and 19.4, of 2000
// of 2048 with 256 experts 15.2 and 14.2.  Workgroups that went through all entries before their own took 4.6 us for 16376
// entries and 7.7 for 32768, at the 18 bytes a cycle that a compute unit takes of a list that is not in its L2 (an empty
// kernel 2.4).
// The first workgroup also writes where the rank's own rows of each local expert begin, behind those of the lower
// source ranks (csrc/kernels/efa_kernels.cu:991-1010).
// ---------------------------------------------------------------------
constexpr int kRankWaves = 8, kRankParts = 4, kRankPart = kRankWaves * kWave;

__global__ __launch_bounds__(kRankPart) void ll_rank_chunk_kernel(
    const int64_t* __restrict__ topk_idx, int n, int num_topk, int num_experts, int32_t* __restrict__ hists,
    RankedBatch batch, const int32_t* __restrict__ recv_count, int num_ranks, int rank, int max_tokens) {
    extern __shared__ u32x2 rank_lds[];  // bytes [E][waves]; int32 [E], what the parts before hold
    static_assert(kRankWaves == 8 && kRankChunkEntries <= kRankParts * kRankPart, "two words of bytes, an entry a lane");
    uint8_t* counts = reinterpret_cast<uint8_t*>(rank_lds);
    int32_t* of_parts = reinterpret_cast<int32_t*>(rank_lds + num_experts);
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block(), b = blockIdx.y;
    const int chunk = int(blockIdx.x) / kRankParts, part = int(blockIdx.x) % kRankParts;
    const int per_chunk = batch.tokens_per_chunk * num_topk;
    const int begin = chunk * per_chunk, end = min(begin + per_chunk, n);
    const int first = begin + part * kRankPart + tid;
    const bool writes_histogram = part == kRankParts - 1;
    if (!writes_histogram && begin + part * kRankPart >= end) return;
    const auto list = entry_list(topk_idx + int64_t(b) * n, n);
    const u32x2 entry = __builtin_amdgcn_raw_buffer_load_b64(list, first * 8, 0, 0);
    u32x2 earlier[kRankParts - 1];
#pragma unroll
    for (int u = 0; u < kRankParts - 1; ++u)
        earlier[u] = __builtin_amdgcn_raw_buffer_load_b64(list, u < part ? (begin + u * kRankPart + tid) * 8 : 0x7ffffff0, 0, 0);
    int own_rows = 0;
    const bool own_wanted = blockIdx.x == 0 && batch.own_first != nullptr && !batch.first_in_finish;
    if (own_wanted) {  // a wave an expert, as far as there are waves
        for (int s = lane; s < rank && w < num_experts / num_ranks; s += kWave) {
            const int c = recv_count[w * num_ranks + s];
            own_rows += c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
        }
    }
    for (int e = tid; e < num_experts; e += kRankPart) rank_lds[e] = u32x2{0u, 0u}, of_parts[e] = 0;
    lds_barrier();
    const uint32_t e = entry[0];
    const bool live = first < end && entry[1] == 0u && e < uint32_t(num_experts);
    uint64_t same = __ballot(live);
    for (int bit = 1; bit < num_experts; bit <<= 1) {
        const bool set = (e & uint32_t(bit)) != 0u;
        const uint64_t votes = __ballot(set);
        same &= set ? votes : ~votes;
    }
    const int lower = __popcll(same & lanes_below(lane));
    if (live && lower == 0) counts[e * kRankWaves + w] = uint8_t(__popcll(same));
#pragma unroll
    for (int u = 0; u < kRankParts - 1; ++u)
        if (u < part && begin + u * kRankPart + tid < end && earlier[u][1] == 0u && earlier[u][0] < uint32_t(num_experts))
            atomicAdd(&of_parts[earlier[u][0]], 1);
    lds_barrier();
    const auto count_before = [&](uint32_t of, int waves) {  // what the parts and waves before have of an expert
        const u32x2 bytes = rank_lds[of];
        uint32_t sum = uint32_t(of_parts[of]);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const int n_bytes = waves - d * 4;
            sum = __builtin_amdgcn_sad_u8(bytes[d] & (n_bytes <= 0 ? 0u : (n_bytes >= 4 ? ~0u : (1u << (n_bytes * 8)) - 1)), 0u, sum);
        }
        return int(sum);
    };
    if (first < end)
        batch.slots[int64_t(b) * batch.stride + first] = live ? count_before(e, w) + lower : -1;
    if (writes_histogram) {
        int32_t* out = hists + int64_t(b) * batch.stride + int64_t(chunk) * num_experts;
        for (int of = tid; of < num_experts; of += kRankPart) out[of] = count_before(uint32_t(of), kRankWaves);
    }
    if (own_wanted) {
        for (int le = w;;) {
            own_rows = wave_inclusive_sum(own_rows);
            if (lane == kWave - 1 && le < num_experts / num_ranks) batch.own_first[le] = own_rows;
            le += kRankWaves;
            if (le >= num_experts / num_ranks) break;
            own_rows = 0;
            for (int s = lane; s < rank; s += kWave) {
                const int c = recv_count[le * num_ranks + s];
                own_rows += c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
            }
        }
    }
}

// The counts of a ranked batch, by one workgroup: columns of the chunk histograms.  By destination, the tables.
__device__ __forceinline__ void ranked_counts(const SendArgs& a, const RankedBatch& batch, int b, int32_t* lds,
                                              int32_t* wave_totals) {
    const int32_t* hists = batch.hists + int64_t(b) * batch.stride;
    const int src_rank = a.src_ranks != nullptr ? a.src_ranks[b] : a.rank;
    for (int e = threadIdx.x; e < a.num_experts; e += block_threads()) {
        const int total = chunk_total(hists, batch.num_chunks, a.num_experts, e);
        if (a.expert_prefix == nullptr) {
            emit_expert_count(e, total, a.num_experts, a.num_ranks, a.rank, src_rank, a.max_tokens, a.recv_count,
                              a.send_count);
        } else {
            lds[e] = total < a.max_tokens ? total : a.max_tokens;
            a.send_count[e] = lds[e];
        }
    }
    if (a.expert_prefix == nullptr) return;
    lds_barrier();
    block_exclusive_scan(lds, a.num_experts, wave_totals);
    by_dest_tables_out(lds, a.num_experts, a.num_ranks, a.by_dest);
}

// Slots within the batch, for batches of many chunks and by-destination ones of many experts: workgroup c adds what the
// chunks before c hold, the last one writes the counts.
__global__ __launch_bounds__(1024) void ll_rank_finish_kernel(SendArgs a, RankedBatch batch) {
    extern __shared__ int32_t before[];  // [E + 1]
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    const int tid = threadIdx.x, threads = block_threads(), c = blockIdx.x, b = blockIdx.y;
    if (c == batch.num_chunks) {
        ranked_counts(a, batch, b, before, wave_totals);
        if (!batch.first_in_finish || c == 0) return;
        __syncthreads();  // the last chunk's histogram has been read; the other workgroups read those before it
        for (int le = tid; le < a.num_experts / a.num_ranks; le += threads) {
            int rows = 0;
            for (int s = 0; s < a.rank; ++s) {
                const int n = a.recv_count[le * a.num_ranks + s];
                rows += n < 0 ? 0 : (n > a.max_tokens ? a.max_tokens : n);
            }
            batch.own_first[le] = rows;
        }
        return;
    }
    const int32_t* hists = batch.hists + int64_t(b) * batch.stride;
    for (int e = tid; e < a.num_experts; e += threads) before[e] = chunk_total(hists, c, a.num_experts, e);
    lds_barrier();
    const int per_chunk = batch.tokens_per_chunk * a.num_topk, n = a.num_tokens * a.num_topk;
    const int end = min((c + 1) * per_chunk, n);
    int32_t* slots = batch.slots + int64_t(b) * batch.stride;
    for (int i = c * per_chunk + tid; i < end; i += threads) {
        int slot = slots[i];
        if (slot < 0) continue;
        slot += before[int(a.topk_idx[int64_t(b) * n + i])];
        slots[i] = slot < a.max_tokens ? slot : -1;
    }
}

// For one wave, from the chunk histograms: the rows of the experts before the lane's `expert` (`first`: an expert's entries
// are clamped to max_tokens) and the entries of the chunks before `chunk` that name it.  Lane l adds up the columns of the
// kPer experts from l * kPer on, whole vectors of them.
template <int kPer>
__device__ __forceinline__ void columns_by_dest(__amdgpu_buffer_rsrc_t hists, int num_chunks, int chunk, int num_experts,
                                                int max_tokens, int expert, int& first, int& below) {
    static_assert(kPer == 1 || kPer == 4, "a word or a vector");
    const int lane = lane_id();
    const bool mine = lane * kPer < num_experts;
    int total[kPer] = {}, lower[kPer] = {};
    constexpr int kAhead = kPer == 1 ? 8 : 4;  // of vectors no more than eight waves a SIMD have registers for
    for (int c0 = 0; c0 < num_chunks; c0 += kAhead) {
        u32x4 v[kAhead];  // zeros past the last histogram
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int at = mine ? ((c0 + u) * num_experts + lane * kPer) * 4 : 0x7ffffff0;
            if constexpr (kPer == 1) v[u][0] = __builtin_amdgcn_raw_buffer_load_b32(hists, at, 0, 0);
            else v[u] = load_row_u32x4<false>(hists, at);
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int i = 0; i < kPer; ++i) total[i] += int(v[u][i]), lower[i] += c0 + u < chunk ? int(v[u][i]) : 0;
    }
    int sum = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) total[i] = total[i] < max_tokens ? total[i] : max_tokens, sum += total[i];
    int run = wave_inclusive_sum(sum) - sum;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int run_of = __shfl(run, expert / kPer, kWave), lower_of = __shfl(lower[i], expert / kPer, kWave);
        if (i == 0 || i <= expert % kPer) first = run_of, below = lower_of;
        run += total[i];
    }
}

// The rows of a ranked batch: a wave's share is a 1 KiB piece as in ll_send_kernel, but nothing is left to be worked out
// by the workgroup, so no wave waits for another.  Selections, places and row are fetched together; behind them, beside
// the row, the columns of the chunks before the token's, shared among the lanes, and a table (the by-destination prefix,
// which without a table are the sums of all columns, or where own rows begin).
// HBM bounds it: 4096 tokens of hidden 7168, top-8, fp8 (302 MB) 52 to 55 us in the kernel trace of a step (5.5 to 5.8 TB/s), 49
// at its fastest, where workgroups that went through the entries of their chunk and shared what they counted, three barriers
// ahead of the stores, took 62; both behind a launch of 4.2.  Called in a row, both launches of a
// send against histograms and that kernel (the ranking's own launch another microsecond slower than now): by destination to
// 8 ranks 4096 tokens 65 -> 59 us, of hidden 1024 23.4 -> 20.7, 2047 tokens of 7168 30.0 -> 29.6, of 4096 with 256 experts
// 26.3 -> 22.9, 1100 23.6 -> 22.5; a dispatch of 4096 tokens 133 -> 125, 2047 70 -> 67.  Two waves a piece, half of the
// stores each: 55 us instead of 50.  With the register allocation left
// open instead of bounded for eight waves a SIMD the same dispatch takes 127, 2047 tokens of 4096 24.4.
// index_rows > 0: the grid has that many rows in front of the token rows whose workgroups build the
// receive side's row index (one (local expert, source) segment each), so that a large one-call
// dispatch needs no launch for it.
template <int kFmt, bool kStream>
__global__ __launch_bounds__(kSendMaxWaves* kWave, 8) void ll_send_ranked_kernel(SendArgs a, DirectOut direct,
                                                                                 RankedBatch batch, FusedIndexArgs index,
                                                                                 int index_rows, int topk_log2) {
    extern __shared__ int32_t ranked_lds[];  // index workgroups: [2 * (E + 1)]; the counting row: [E + 1]
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    // First the index rows (started first, so that their few microseconds of scans run beside the token rows instead
    // of behind them), then one row per token, then the counting row.
    const int t = int(blockIdx.y) - index_rows, b = blockIdx.z;
    if (t < 0) {
        const int seg = int(blockIdx.y) * int(gridDim.x) + int(blockIdx.x);
        if (seg < index.num_local_experts * index.num_ranks) recv_index_block(index, seg, ranked_lds, wave_totals);
        return;
    }
    if (t == a.num_tokens) {
        if (blockIdx.x == 0) ranked_counts(a, batch, b, ranked_lds, wave_totals);
        return;
    }
    const int lane = lane_id(), num_topk = a.num_topk, num_experts = a.num_experts;
    const int item = int(blockIdx.x) * (block_threads() >> 6) + wave_in_block();
    if (item >= (a.pieces_per_row << a.split_log2)) return;
    const int split = 1 << a.split_log2, part = item & (split - 1), piece = item >> a.split_log2;
    const int64_t row_id = int64_t(b) * a.num_tokens + t;
    const auto token_row = row_buffer(a.x + uint64_t(row_id) * (uint32_t(a.hidden) * 2), a.hidden * 2);
    u32x4 lo, hi = {0u, 0u, 0u, 0u};  // zeros past the row's end
    if constexpr (kFmt == kRowBF16) {
        lo = load_row_u32x4<false>(token_row, piece * 1024 + lane * 16);
    } else {
        lo = load_row_u32x4<false>(token_row, piece * 2048 + lane * 32);
        hi = load_row_u32x4<false>(token_row, piece * 2048 + lane * 32 + 16);
    }
    // Selection k in the lanes k, k + 2^topk_log2, ...: 2^topk_log2 >= K, so that the lanes share a selection's columns.
    const int k = lane & ((1 << topk_log2) - 1);
    int expert = 0, slot = -1;
    if (k < num_topk) {
        slot = batch.slots[int64_t(b) * batch.stride + int64_t(t) * num_topk + k];
        expert = int(a.topk_idx[row_id * num_topk + k]);
    }
    if (slot < 0) expert = 0;
    int first = 0;  // by destination: where the expert's run of rows begins in the send buffer
    const bool by_dest = a.expert_prefix != nullptr;
    if (batch.in_full) {
        if (by_dest) first = a.expert_prefix[expert];
    } else {
        const int chunk = batch.chunk_of(t);
        const auto hists = row_buffer(reinterpret_cast<const uint8_t*>(batch.hists + int64_t(b) * batch.stride),
                                      batch.num_chunks * num_experts * 4);
        int below = 0;
        if (by_dest) {
            if (num_experts <= kWave) columns_by_dest<1>(hists, batch.num_chunks, chunk, num_experts, a.max_tokens, expert, first, below);
            else columns_by_dest<4>(hists, batch.num_chunks, chunk, num_experts, a.max_tokens, expert, first, below);
        } else {
            const int step = kWave >> topk_log2;
            for (int c = lane >> topk_log2; c - (lane >> topk_log2) < chunk; c += 4 * step) {
                int v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    v[u] = int(__builtin_amdgcn_raw_buffer_load_b32(
                        hists, c + u * step < chunk ? ((c + u * step) * num_experts + expert) * 4 : 0x7fffffff, 0, 0));
#pragma unroll
                for (int u = 0; u < 4; ++u) below += v[u];
            }
            for (int d = 1 << topk_log2; d < kWave; d <<= 1) below += __shfl_xor(below, d, kWave);
        }
        if (slot >= 0) slot += below;
        if (slot >= a.max_tokens) slot = -1;
        if (item == 0 && lane < num_topk && a.pair_slot != nullptr) a.pair_slot[int64_t(t) * num_topk + lane] = slot;
    }
    const int src_rank = a.src_ranks != nullptr ? a.src_ranks[b] : a.rank;
    const int64_t data_bytes = row_data_bytes(a.hidden, kFmt), scale_bytes = row_scale_bytes(a.hidden, kFmt);
    const int64_t stride = row_stride_bytes(a.hidden, kFmt);
    uint8_t *row = nullptr, *scale_row = nullptr;
    if (slot >= 0 && lane < num_topk) {
        // expert / E_l by multiply-high; magic 0 stands for E_l == 1
        const int dst_rank = a.rank_of_expert_magic != 0 ? int(__umulhi(uint32_t(expert), a.rank_of_expert_magic)) : expert;
        const int local = expert - dst_rank * (num_experts / a.num_ranks);
        if (by_dest) {
            row = a.send_slots + (int64_t(first) + slot) * stride;
        } else if (dst_rank != a.rank) {
            if (a.send_slots != nullptr) row = a.send_slots + (int64_t(expert) * a.max_tokens + slot) * stride;
        } else if (direct.packed_x == nullptr) {
            row = a.recv_staging + ((int64_t(local) * a.num_ranks + src_rank) * a.max_tokens + slot) * stride;
        }
        if (row != nullptr) {
            scale_row = row + align16(data_bytes);
            if (item == 0) {
                const u32x4 tail = {uint32_t(t), uint32_t(lane), uint32_t(src_rank), uint32_t(local)};
                *reinterpret_cast<u32x4*>(scale_row + align16(scale_bytes)) = tail;
            }
        } else if (dst_rank == a.rank) {
            const int64_t out_row = int64_t(local) * a.num_ranks * a.max_tokens + batch.own_first[local] + slot;
            row = direct.packed_x + out_row * data_bytes;
            scale_row = direct.packed_scales + out_row * scale_bytes;
            if (item == 0) direct.src_info[out_row] = t;
        }
    }
    u32x4 payload = lo;
    uint32_t scale_bits = 0;
    int scale_off = 0x7fffffff;
    if constexpr (kFmt != kRowBF16) {
        payload = quantise_16<kFmt>(lo, hi, scale_bits);
        const int group = piece * 8 + (lane >> 3);
        if ((lane & 7) == 0 && group < a.hidden / kGroup) scale_off = kFmt == kRowFP8UE8M0 ? group : group * 4;
    }
    store_selections<kFmt, kStream>(reinterpret_cast<uint64_t>(row), reinterpret_cast<uint64_t>(scale_row), num_topk, part,
                                    split, int(data_bytes), int(scale_bytes), piece * 1024 + lane * 16, payload, scale_off,
                                    scale_bits);
}

// ---------------------------------------------------------------------
// Receive side.  Every copying wave rebuilds the segment prefix from the E
// counts (a few hundred ints) in its registers, then walks the flat row index
// space: row -> (segment, j) by ballot, one wave per row part.
// Ranges are the reference's: inside an expert's packed range the source ranks
// come in ascending order, begin(e, s) = sum of cnt(e, s') over s' < s
// (csrc/kernels/efa_kernels.cu:991-1010, :1031-1050); the slot order inside a
// segment is fixed by the staging order, not by atomics (:1059-1213 is the
// reference's deterministic scatter).
//
// own_rank >= 0 (one-call dispatch): the rows this rank sends to its own
// experts are not in the staging area — the send side puts them straight into
// the packed tensors, behind the rows of the lower ranks — so the copying waves
// skip the own segments and move the segments of the higher ranks up by the
// expert's own count.  With own_entries >= 0 (single launch) that count is
// recounted from the rank's own indices, because the launch that reads
// recv_count's own entries is the one that writes them; with kOwnCounted (the
// send kernel has finished) recv_count holds it.  It takes a value of its own to
// say so: the list of a rank without tokens is empty, and its address may be null.
// ---------------------------------------------------------------------
struct RecvArgs {
    const uint8_t* recv_staging;
    const int32_t* recv_count;
    int hidden, num_local_experts, num_ranks, max_tokens, fmt, parts_log2;
    RankDivider expert_of;
    uint8_t* packed_x;
    uint8_t* packed_scales;
    int32_t* src_info;
    int64_t* layout_range;
    int32_t* packed_count;
    int32_t* stats;
    ObservedRows observed;
};

__device__ __forceinline__ int clamp_count(int c, int max_tokens) {
    return c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
}

// own_cnt[e_l] (LDS, unclamped) = rows this rank sends to its own expert e_l, counted by the whole
// workgroup in two steps so that other loads can be issued in between: `begin` issues the first index
// loads and clears the counters, `finish` counts and ends with a barrier.
constexpr int kOwnAhead = 4;  // index loads in flight per thread, two entries each
constexpr int kOwnCounted = -1;

struct OwnCountLoads {
    EntryPair v[kOwnAhead];
};

__device__ __forceinline__ void own_row_counts_begin(const RecvArgs& a, const int64_t* own_topk, int own_entries,
                                                     int32_t* own_cnt, OwnCountLoads& loads) {
    const int tid = threadIdx.x, threads = block_threads();
    if (own_entries == kOwnCounted) return;
    const auto list = entry_list(own_topk, own_entries);
#pragma unroll
    for (int r = 0; r < kOwnAhead; ++r) loads.v[r].load(list, tid + r * threads);
    for (int le = tid; le < a.num_local_experts; le += threads) own_cnt[le] = 0;
    lds_barrier();
}

__device__ __forceinline__ void own_row_counts_finish(const RecvArgs& a, const int64_t* own_topk, int own_entries,
                                                      int own_rank, int32_t* own_cnt, OwnCountLoads& loads) {
    const int tid = threadIdx.x, threads = block_threads();
    if (own_entries == kOwnCounted) {
        for (int le = tid; le < a.num_local_experts; le += threads)
            own_cnt[le] = a.recv_count[le * a.num_ranks + own_rank];
        lds_barrier();
        return;
    }
    const auto list = entry_list(own_topk, own_entries);
    const uint32_t first = uint32_t(own_rank) * a.num_local_experts;
    for (int base = 0;;) {
#pragma unroll
        for (int r = 0; r < kOwnAhead; ++r)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                uint32_t le;
                if (loads.v[r].expert(i, first, uint32_t(a.num_local_experts), le) &&
                    (base + tid + r * threads) * 2 + i < own_entries)
                    atomicAdd(&own_cnt[le], 1);
            }
        base += kOwnAhead * threads;
        if (base * 2 >= own_entries) break;
#pragma unroll
        for (int r = 0; r < kOwnAhead; ++r) loads.v[r].load(list, base + tid + r * threads);
    }
    lds_barrier();
}

constexpr int kRecvDepth = 4;  // 16-byte loads in flight per lane

// One unit of the copying waves' work: a run of 16-byte vectors of one staged row.
template <bool kStream>
struct RecvItem {
    const uint8_t* src;
    int le, source, slot;  // slot: the row's place among the rows copied for the expert, own rows not counted
    int v_begin;
    bool carries_tail;  // also moves the row's scales and source index
    RowPart<kRecvDepth, false, kStream> payload;
    uint32_t scale;  // a lane's scale word, with the tail
    int32_t info;
};

// Workgroups [0, num_copy_blocks) copy rows; workgroup num_copy_blocks writes layout_range,
// packed_count and stats and copies nothing.  A copying wave builds the segment prefix in its own
// registers (WaveSegments) from the E counts.  Where a row lands may depend on the own count of its
// expert, where it comes from does not: a wave issues the loads of its first item before the
// workgroup settles the own counts.
// lds: [num_segments + 1 + num_local_experts] ints; wave_totals: 16 ints.
template <int kPer, bool kStream>
__device__ __forceinline__ void recv_rows_impl(const RecvArgs& a, int block, int num_copy_blocks,
                                               const int64_t* own_topk, int own_entries, int own_rank, int32_t* lds,
                                               int32_t* wave_totals) {
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block();
    const int threads = block_threads(), waves = threads >> 6;
    const int num_ranks = a.num_ranks, max_tokens = a.max_tokens;
    const int num_segments = a.num_local_experts * num_ranks;
    const bool own_placed = own_rank >= 0;
    OwnCountLoads own_loads;

    if (block == num_copy_blocks) {  // the metadata workgroup
        int32_t* own_cnt = lds + num_segments + 1;
        if (own_placed) {
            own_row_counts_begin(a, own_topk, own_entries, own_cnt, own_loads);
            own_row_counts_finish(a, own_topk, own_entries, own_rank, own_cnt, own_loads);
        }
        for (int s = tid; s < num_segments; s += threads) {
            const int le = s / num_ranks;
            const bool own = own_placed && s - le * num_ranks == own_rank;
            lds[s] = clamp_count(own ? own_cnt[le] : a.recv_count[s], max_tokens);
        }
        lds_barrier();
        block_exclusive_scan(lds, num_segments, wave_totals);
        if (tid == 0) report_observed(a.observed, lds[num_segments]);
        for (int s = tid; s < num_segments; s += threads) {
            const int le = s / num_ranks;
            const int64_t cnt = lds[s + 1] - lds[s];
            const int64_t begin = lds[s] - lds[le * num_ranks];
            a.layout_range[s] = cnt > 0 ? ((begin << 32) | cnt) : 0;
        }
        for (int le = tid; le < a.num_local_experts; le += threads) {
            const int c = lds[(le + 1) * num_ranks] - lds[le * num_ranks];
            a.packed_count[le] = c;
            if (a.stats != nullptr) a.stats[le] += c;
        }
        return;
    }

    int32_t* own_cnt = lds;  // [E_l]
    WaveSegments<kPer> seg_table;
    DEEPEP_PHASE(0);
    if (own_placed) own_row_counts_begin(a, own_topk, own_entries, own_cnt, own_loads);
    wave_load_int32<kPer>(a.recv_count, num_segments, lane, seg_table.cnt);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        seg_table.aux[u] = 0;
        seg_table.cnt[u] = clamp_count(seg_table.cnt[u], max_tokens);
    }
    if (own_placed) {  // the own segments (le * R + own_rank) hold nothing to copy
        int source = lane * kPer - a.expert_of(lane * kPer) * num_ranks;  // source rank of this lane's first segment
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (source == own_rank) seg_table.cnt[u] = 0;
            source = source + 1 == num_ranks ? 0 : source + 1;
        }
    }
    wave_segments_finish(seg_table);
    DEEPEP_PHASE(1);

    const uint32_t data_bytes = uint32_t(row_data_bytes(a.hidden, a.fmt));
    const uint32_t data_pad = uint32_t(align16(data_bytes));
    const uint32_t scale_bytes = uint32_t(row_scale_bytes(a.hidden, a.fmt));
    const uint32_t stride = uint32_t(row_stride_bytes(a.hidden, a.fmt));
    const int slots_per_expert = max_tokens * num_ranks;
    const int waves_total = num_copy_blocks * waves;
    const int num_vec = int(data_bytes / 16);
    const int parts = 1 << a.parts_log2;
    const int num_items = seg_table.total << a.parts_log2;

    // What the tail-carrying part of a row moves besides payload: one scale word per lane (the first 64;
    // a wider row's remainder is copied after the stores) and, in lane 0, the source index.  They are
    // loaded with the payload, not behind its stores: one round trip per row instead of two.
    const int scale_dwords = int(scale_bytes / 4);
    const bool has_scales = a.packed_scales != nullptr && scale_dwords > 0;
    auto load_first = [&](int item, RecvItem<kStream>& it) {
        const int row = item >> a.parts_log2, part = item & (parts - 1);
        int seg_first, unused, v_end;
        const int seg = wave_segments_find(seg_table, row, seg_first, unused);
        it.le = a.expert_of(seg);
        it.source = seg - it.le * num_ranks;
        it.src = a.recv_staging + uint64_t(uint32_t(seg * max_tokens + (row - seg_first))) * stride;
        row_part_range(num_vec, a.parts_log2, part, it.v_begin, v_end);
        it.payload.load(it.src, it.v_begin, v_end, lane);
        it.carries_tail = part == parts - 1;  // the last part is the shortest
        it.scale = 0, it.info = 0;
        if (it.carries_tail) {
            if (has_scales && lane < scale_dwords) it.scale = reinterpret_cast<const uint32_t*>(it.src + data_pad)[lane];
            if (lane == 0) it.info = *reinterpret_cast<const int32_t*>(it.src + data_pad + uint32_t(align16(scale_bytes)));
        }
        it.slot = row - wave_segments_prefix(seg_table, it.le * num_ranks);
    };
    auto finish = [&](RecvItem<kStream>& it) {
        int slot = it.slot;
        if (own_placed && it.source > own_rank)
            slot += clamp_count(__builtin_amdgcn_readfirstlane(own_cnt[it.le]), max_tokens);
        const uint32_t out_row = uint32_t(it.le * slots_per_expert + slot);
        it.payload.store(a.packed_x + uint64_t(out_row) * data_bytes, it.v_begin, lane);
        if (!it.carries_tail) return;
        if (has_scales) {
            const uint32_t* s32 = reinterpret_cast<const uint32_t*>(it.src + data_pad);
            uint32_t* d32 = reinterpret_cast<uint32_t*>(a.packed_scales + uint64_t(out_row) * scale_bytes);
            if (lane < scale_dwords) d32[lane] = it.scale;
            for (int v = kWave + lane; v < scale_dwords; v += kWave) d32[v] = s32[v];
        }
        if (lane == 0) a.src_info[out_row] = it.info;
    };

    RecvItem<kStream> it;
    int item = block * waves + w;
    const bool have_first = item < num_items;
    if (have_first) {
        DEEPEP_PHASE(2);
        load_first(item, it);
    }
    // every wave of the workgroup passes here, with or without rows to copy
    if (own_placed) own_row_counts_finish(a, own_topk, own_entries, own_rank, own_cnt, own_loads);
    if (have_first) {
        finish(it);
        DEEPEP_PHASE(3);
        item += waves_total;
    }
    for (; item < num_items; item += waves_total) {
        load_first(item, it);
        finish(it);
    }
}

template <bool kStream>
__device__ __forceinline__ void recv_rows(const RecvArgs& a, int block, int num_copy_blocks, const int64_t* own_topk,
                                          int own_entries, int own_rank, int32_t* lds, int32_t* wave_totals) {
    if (a.num_local_experts * a.num_ranks <= 4 * kWave)
        recv_rows_impl<4, kStream>(a, block, num_copy_blocks, own_topk, own_entries, own_rank, lds, wave_totals);
    else
        recv_rows_impl<16, kStream>(a, block, num_copy_blocks, own_topk, own_entries, own_rank, lds, wave_totals);
}

// own_rank >= 0: the send side has already put this rank's own rows at their packed position.
__global__ __launch_bounds__(256) void ll_recv_kernel(RecvArgs a, int own_rank) {
    extern __shared__ int32_t flat[];  // [num_segments + 1 + E_l]
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    recv_rows<false>(a, blockIdx.x, int(gridDim.x) - 1, nullptr, kOwnCounted, own_rank, flat, wave_totals);
}

// ---------------------------------------------------------------------
// Single-launch dispatch for small batches (dispatch_in_one_launch()): the send
// workgroups, the counting workgroup and the receive workgroups of the two
// kernels above in one grid.  No workgroup waits on another: the receive
// workgroups copy only the peers' rows (already in the staging area when the
// launch starts); the send workgroups place the rank's rows for its own
// experts at their final packed position, which they find from the lower
// ranks' counts, and the receive workgroups make room for them by recounting
// them from the rank's own indices.  The packed ranges are the reference's
// (ascending source rank, csrc/kernels/efa_kernels.cu:991-1010).
// (The reference's dispatch is one kernel with a send and a receive phase as
// well: csrc/kernels/coop_dispatch_send.cuh:304, coop_dispatch_recv.cuh:42.)
// ---------------------------------------------------------------------
template <int kFmt, bool kStream, bool kMany>
__global__ __launch_bounds__(kSendMaxWaves* kWave) void ll_dispatch_fused_kernel(SendArgs sa, RecvArgs ra, int blocks_per_token,
                                                                                 int num_send_blocks) {
    extern __shared__ int32_t dyn_lds[];  // counting: [E]; receive: [segments + 1 + E_l]
    __shared__ SendLds lds;
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    const int block = blockIdx.x;
    if (block < num_send_blocks) {
        const DirectOut direct = {ra.packed_x, ra.packed_scales, ra.src_info};
        if constexpr (kMany)
            send_token_block<kFmt, kStream, false, true>(sa, direct, 0, block * sa.tokens_per_block, 0, lds, dyn_lds);
        else
            send_token_block<kFmt, kStream, false, false>(sa, direct, 0, block / blocks_per_token, block % blocks_per_token,
                                                          lds, dyn_lds);
    } else if (block == num_send_blocks) {
        send_count_block(sa, 0, dyn_lds);
    } else {
        recv_rows<kStream>(ra, block - num_send_blocks - 1, int(gridDim.x) - num_send_blocks - 2, sa.topk_idx,
                  sa.num_tokens * sa.num_topk, sa.rank, dyn_lds, wave_totals);
    }
}

// Experts whose columns a wave adds up: a word a lane, or a vector.
static bool columns_by_dest_fit(int num_experts) {
    return num_experts <= kWave || (num_experts <= 4 * kWave && num_experts % 4 == 0);
}

// Whether a by-destination send (what an all-to-all ships: one contiguous message per peer) of up to 8192 entries makes
// its tables itself -- send_count[e], clamped to the M slots of a pair, its exclusive prefix over the experts, which is the
// first row of every expert's run, and the per-rank counts and prefix the transport cuts the buffer by; reference: the
// count + prefix phases of ll_dispatch_route_and_pack_v3 (csrc/kernels/efa_kernels.cu:2358-2371: ll_dispatch_count_kernel,
// prefix_sum_kernel).  Every token's workgroup then goes through the whole batch instead of half of it, and one wave
// through the experts: up to 1024 experts that costs less than a launch ahead, past them only for batches of up to 2048
// entries.  Microseconds of the send with the tables made by itself against a launch before it, top-8, fp8:
//   300 tokens, 64 experts, hidden 7168      10.7 / 13.5        300 tokens, 256 experts, hidden 2048      6.0 /  8.6
//   1024 tokens, 64 experts, hidden 7168     18.2 / 19.5        1000 tokens, 1024 experts, hidden 2048   12.1 / 14.3
//   1000 tokens, 4096 experts, hidden 2048   20.1 / 15.3
// Both counts of an expert share a 32-bit word: fewer than 2^16 entries.
constexpr int kByDestInBlockExperts = 1024, kByDestInBlockEntries = 2048;
static bool by_dest_tables_in_send(int n, int num_experts) {
    return n <= kSelfRankMaxEntries && (num_experts <= kByDestInBlockExperts || n <= kByDestInBlockEntries);
}

// ---------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------
static int check_ll_shape(int num_tokens, int hidden, int num_topk, int num_experts, int num_ranks, int rank,
                          int max_tokens, int row_format) {
    EP_HOST_ASSERT(num_tokens >= 0 && hidden > 0 && num_topk > 0 && num_topk <= kMaxTopk);
    EP_HOST_ASSERT(hidden % 128 == 0);
    EP_HOST_ASSERT(num_ranks > 0 && num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(rank >= 0 && rank < num_ranks);
    EP_HOST_ASSERT(max_tokens > 0 && num_tokens <= max_tokens);
    EP_HOST_ASSERT(row_format >= kRowBF16 && row_format <= kRowFP8UE8M0);
    EP_HOST_ASSERT(row_format != kRowFP8UE8M0 || (hidden / 128) % 4 == 0);
    EP_HOST_ASSERT(int64_t(num_tokens) * num_topk < (int64_t(1) << 30));
    EP_HOST_ASSERT(num_experts <= 4096);
    return 0;
}

// Waves that a token's row takes.
static int row_pieces(int hidden, int row_format) {
    return row_format == kRowBF16 ? (hidden * 2 + 1023) / 1024 : (hidden / kGroup + 7) / 8;
}

// Tokens of a workgroup that ranks its own slots, of `items` waves each (kManyBlocks says why).
static int tokens_per_send_block(int items, int max_waves, int num_topk, int num_tokens) {
    int tokens = 1;
    while (tokens < 4 && 2 * tokens * items <= max_waves && 2 * tokens * num_topk <= kWave &&
           num_tokens >= 2 * tokens * kManyBlocks)
        tokens *= 2;
    return tokens;
}

constexpr int kFusedMaxWaves = 8, kFusedManyPieces = 2, kFusedEvenEntries = 1792;
constexpr int kFusedFewFrom = 4608, kFusedFewTokens = 1536;  // entries, tokens

// Whether a one-call dispatch runs as one launch: up to 8192 entries and rows always.  Past them it saves a launch or two
// (4 to 8 us) and pays with its workgroups' sweeps through the entries, fewer of them where a workgroup has several
// tokens, and with copying waves that go round for more rows, which falls behind the flat copy once the rows are large in
// all.  Microseconds of a step, top-8 unless said, fp8 unless said, three launches / one, by the millions of entries that
// the send workgroups go through and the MB of rows expected:
//   1100 x 2048   2.4   19   44.8 / 39.5     1100 x 2048 bf16   9.7   36   51.5 / 43.9     1100 x 7168  9.7   66  106.8 / 103.5
//   2300 x 2048  10.6   39   73.3 / 66.3     2000 x 2048 bf16, top-6                       2000 x 4096  32    69  112.1 / 112.1
//   3400 x 2048  23     58  100.1 / 99.5                       24    49   64.1 / 57.7      1500 x 7168  18    90  140.5 / 142.8
//   4096 x 2048  33.5   70  115.4 / 114.0    3000 x 2048 bf16, top-6                       1500 x 5120 bf16
//   1700 x 4096  23     58  100.7 / 94.0                       54    74   84.8 / 90.3                   18   123  127.7 / 140.0
// The rank of the hottest of 256 experts on 64 ranks: 100 tokens of 4096 86.2 / 77.4, 200 of 2048 86.7 / 80.2.
// One workgroup counts all entries, one a thread and round, and the launch waits for it: 96 rounds at most, and 44 for rows of
// one wave, whose launches are short.  Those also have more sweeps for their bytes, and so does a token of more than 32
// selections.  Microseconds of the dispatch alone, three launches / one:
//   rows of one wave    1375 x 512 13.2 / 11.5    1750 x 512 bf16 16.5 / 17.2    2200 x 512 16.4 / 18.5    3500 x 128 bf16 17.7 / 25.8
//     top-2, 5000 x 512 14.3 / 13.7 (12.5 M), 5500 15.0 / 15.3 (15 M)    top-64, 129 x 512 14.5 / 15.9, 257 x 1024 21.9 / 22.5
//   top-32, 750 x 2048 36.1 / 34.5 (94 rounds), 1000 43.5 / 49.3 (125)   top-16, 2000 x 2048 42.5 / 33.6 (62, in eight waves)
//   top-64 in rows of 1152 to 2048 bytes, 131 tokens 16.6 / 17.8 and 20.3 / 19.1
//   rows of 256 bytes, some 66000 29.4 / 23.4, 116000 39.5 / 42.4
static bool dispatch_in_one_launch(int num_tokens, int num_topk, int num_experts, int max_tokens, int hidden,
                                   int row_format, int64_t expected_rows) {
    if (deepep_ll_dispatch_is_single_launch(num_tokens, num_topk, num_experts, max_tokens, expected_rows) != 0) return true;
    const int pieces = row_pieces(hidden, row_format);
    const int tokens = pieces <= kFusedManyPieces ? tokens_per_send_block(pieces, kFusedMaxWaves, num_topk, num_tokens) : 1;
    const int64_t entries = int64_t(num_tokens) * num_topk;
    const int64_t send_blocks = (num_tokens + tokens - 1) / tokens * int64_t((pieces + kFusedMaxWaves - 1) / kFusedMaxWaves);
    const int counting_threads = (pieces * tokens <= 4 ? 4 : kFusedMaxWaves) * kWave;
    if (num_topk > 32 && row_data_bytes(hidden, row_format) < 2048) return false;
    const int64_t rows = estimated_rows(expected_rows, num_experts, max_tokens);
    return entries <= int64_t(pieces == 1 ? 44 : 96) * counting_threads &&
           send_blocks * entries <= (int64_t(pieces == 1 ? 14 : 24) << 20) && rows <= 96 * 1024 &&
           rows * row_payload_bytes(hidden, row_format) <= (int64_t(72) << 20);
}

static int launch_send_side(const void* x, const int64_t* topk_idx, const int32_t* src_ranks, int num_src,
                            int num_tokens, int hidden, int num_topk, int num_experts, int num_ranks, int rank,
                            int max_tokens, int row_format, void* recv_staging, int32_t* recv_count,
                            void* send_slots, int32_t* send_count, int32_t* pair_slot, void* workspace,
                            size_t workspace_bytes, hipStream_t stream, const RecvArgs* fused_recv = nullptr,
                            int64_t fused_recv_wave_items = 0, const DirectOut* own_rows_direct = nullptr,
                            const ByDestTables* by_dest = nullptr, FusedIndexArgs* fused_index = nullptr,
                            bool* index_was_fused = nullptr) {
    const int n = num_tokens * num_topk;
    // How slots get ranked: the launch that stores the rows does it for itself while it is the only one and has no more
    // than kSelfRankMaxEntries entries to go through.
    const bool prefix_in_block = by_dest != nullptr && by_dest_tables_in_send(n, num_experts);
    bool ranked = fused_recv == nullptr && (n > kSelfRankMaxEntries || own_rows_direct != nullptr ||
                                            (by_dest != nullptr && !prefix_in_block));
    const int64_t hist_bytes = chunk_hist_bytes(num_tokens, num_topk, num_experts);
    const int64_t slot_bytes = align256(int64_t(n) * 4);
    int64_t first_bytes = own_rows_direct != nullptr ? align256(int64_t(num_experts) * 4) : 0;
    // What the chunks before a token's hold of its experts is added up by the waves that store its rows, up to
    // kSendColumns of them and, by destination, up to 256 experts; otherwise, and without room for slots that nobody sees,
    // by a launch between the two.
    RankedBatch batch = {};
    batch.tokens_per_chunk = rank_chunk_tokens(num_topk);
    batch.num_chunks = (num_tokens + batch.tokens_per_chunk - 1) / batch.tokens_per_chunk;
    batch.chunk_of = make_rank_divider(batch.tokens_per_chunk);
    // A workspace may hold the histograms alone.  The slots then go where the caller wants them and where own rows begin over a
    // histogram that has been read; sends whose slots nobody wants rank themselves, whatever that takes.
    const bool room = workspace_bytes >= size_t(hist_bytes + first_bytes + slot_bytes) * size_t(num_src);
    if (!room && pair_slot == nullptr) ranked = false;
    if (!room && own_rows_direct != nullptr) first_bytes = 0, batch.first_in_finish = 1;
    batch.in_full = batch.num_chunks > kSendColumns || (by_dest != nullptr && !columns_by_dest_fit(num_experts)) || !room;
    const bool slots_in_scratch = !batch.in_full || pair_slot == nullptr;
    const int64_t scratch_bytes = hist_bytes + first_bytes + (slots_in_scratch ? slot_bytes : 0);
    EP_HOST_ASSERT(workspace != nullptr && workspace_bytes >= size_t(ranked ? scratch_bytes : hist_bytes) * size_t(num_src));
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(workspace) & 15) == 0);
    EP_HOST_ASSERT(by_dest == nullptr || (num_src == 1 && src_ranks == nullptr && fused_recv == nullptr &&
                                          own_rows_direct == nullptr));
    // own_rows_direct (the form of the one-call dispatch in more than one launch): as in the single launch, the rows
    // for this rank's own experts go straight to their packed position behind the lower ranks' rows
    EP_HOST_ASSERT(own_rows_direct == nullptr || (num_src == 1 && src_ranks == nullptr));
    EP_HOST_ASSERT(num_tokens < 65535 && num_src <= 65535);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    if (ranked) {
        batch.hists = reinterpret_cast<int32_t*>(ws);
        if (batch.first_in_finish)
            batch.own_first = reinterpret_cast<int32_t*>(ws) + int64_t(std::max(batch.num_chunks - 1, 0)) * num_experts;
        else if (own_rows_direct != nullptr)
            batch.own_first = reinterpret_cast<int32_t*>(ws + hist_bytes);
        batch.slots = slots_in_scratch ? reinterpret_cast<int32_t*>(ws + hist_bytes + first_bytes) : pair_slot;
        batch.stride = scratch_bytes / 4;
        if (batch.num_chunks > 0) {
            launch(ll_rank_chunk_kernel, dim3(batch.num_chunks * kRankParts, num_src), kRankPart,
                                   size_t(num_experts) * (kRankWaves + sizeof(int32_t)), stream,
                topk_idx, n, num_topk, num_experts, reinterpret_cast<int32_t*>(ws), batch, recv_count, num_ranks, rank,
                max_tokens);
            EP_LAUNCH_CHECK();
        }
    }

    const int pieces = row_pieces(hidden, row_format);
    // A small batch cannot fill 1024 SIMDs with one wave per row piece: give a share of the
    // K stores of each piece to a second wave.
    int split_log2 = int64_t(num_src) * num_tokens * pieces < 4096 && num_topk > 1 ? 1 : 0;
    // In the single launch the receive workgroups share the chip: whole tokens per workgroup, and
    // workgroups small enough that two fit a compute unit.
    if (fused_recv != nullptr) split_log2 = 0;
    const int items = pieces << split_log2;  // waves per token
    const int max_waves = fused_recv != nullptr ? kFusedMaxWaves : kSendMaxWaves;
    int waves = items < max_waves ? items : max_waves;
    const int blocks_per_token = (items + waves - 1) / waves;
    // Every workgroup of the single launch goes through the batch's entries, the send ones for their slots and the
    // receive ones for the own counts: from some 1500 entries on the eighth wave that a 7168-wide row has no piece
    // for is worth its place (256 tokens, top-8 15.9 -> 15.1 us, 1024 tokens 40.9 -> 39.6; 128 tokens 8.0 -> 8.1).
    if (fused_recv != nullptr && n > 1536 && waves > 4) waves = 8;
    // A row of several workgroups is cut evenly in the single launch where that does without two waves or more of each: the
    // waves that have no piece take others' places on the chip.  Past 1792 entries a step has lost by it, in other worlds than
    // those in which it gained below; the dispatch alone gains past them too (300 x 5120 to 8 13.9 / 12.9, 400 at top-6 13.8 /
    // 12.1, 1000 41.3 / 39.9; 260 x 6144 12.7 / 13.4).  Microseconds of a step in bf16, eight waves / five (six at hidden 6144), top-8 to 32 ranks:
    //   100 x 5120 to 8    16.7 / 16.2    128 x 5120  21.8 / 20.6    180 to 16  28.0 / 26.3    220  30.6 / 29.5
    //   190 x 4608 to 64   28.8 / 27.3    150 x 6144  27.6 / 26.6    16 and 60  12.2 and 14.4 either way
    //   250 x 5120 to 64   28.1 / 28.7    400 to 8    39.0 / 39.9    1000 to 8  91.0 / 92.7; seven of eight, 128 x 7168 26.7 / 27.0
    const int even_waves = (items + blocks_per_token - 1) / blocks_per_token;
    if (fused_recv != nullptr && blocks_per_token > 1 && n <= kFusedEvenEntries && even_waves + 2 <= waves) waves = even_waves;
    if (fused_recv != nullptr && waves < 4) waves = 4;  // the receive workgroups want a few waves each
    int tokens_per_block = 1;
    if (!ranked && blocks_per_token == 1 && (fused_recv == nullptr || items <= kFusedManyPieces))
        tokens_per_block = tokens_per_send_block(items, max_waves, num_topk, num_tokens);
    if (fused_recv == nullptr && 2 * items > 8 &&
        (n < kTwoTokensFrom || num_tokens < 4 * kManyBlocks || (items > 6 && (items != 8 || by_dest == nullptr))))
        tokens_per_block = 1;
    const int token_blocks = (num_tokens + tokens_per_block - 1) / tokens_per_block;
    if (tokens_per_block > 1) waves = std::max(waves, items * tokens_per_block);
    // floor(e / E_l) == umulhi(e, ceil(2^32 / E_l)) for every e below 2^16.
    const uint32_t experts_per_rank = uint32_t(num_experts / num_ranks);
    const uint32_t magic =
        experts_per_rank == 1 ? 0u : uint32_t(((uint64_t(1) << 32) + experts_per_rank - 1) / experts_per_rank);
    EP_HOST_ASSERT(num_experts < 65536);
    SendArgs sa;
    sa.x = reinterpret_cast<const uint8_t*>(x);
    sa.topk_idx = topk_idx;
    sa.src_ranks = src_ranks;
    sa.num_tokens = num_tokens, sa.hidden = hidden, sa.num_topk = num_topk, sa.num_experts = num_experts;
    sa.num_ranks = num_ranks, sa.rank = rank, sa.max_tokens = max_tokens;
    sa.pieces_per_row = pieces, sa.split_log2 = split_log2;
    sa.tokens_per_block = tokens_per_block, sa.token_of = make_rank_divider(num_topk);
    sa.rank_of_expert_magic = magic;
    sa.recv_staging = reinterpret_cast<uint8_t*>(recv_staging);
    sa.send_slots = reinterpret_cast<uint8_t*>(send_slots);
    sa.pair_slot = pair_slot, sa.recv_count = recv_count, sa.send_count = send_count;
    sa.expert_prefix = by_dest != nullptr ? by_dest->expert_prefix : nullptr;
    sa.prefix_in_block = prefix_in_block ? 1 : 0;
    sa.by_dest = by_dest != nullptr ? *by_dest : ByDestTables{nullptr, nullptr, nullptr};
    if (ranked && batch.in_full) {
        launch(ll_rank_finish_kernel, dim3(batch.num_chunks + 1, num_src), 1024, size_t(num_experts + 1) * sizeof(int32_t), stream,
            sa, batch);
        EP_LAUNCH_CHECK();
    }

    if (fused_recv != nullptr) {  // single launch: send workgroups, the counting workgroup, receive workgroups
        EP_HOST_ASSERT(num_src == 1 && src_ranks == nullptr);
        const int num_send_blocks = blocks_per_token * token_blocks;
        int64_t fused_recv_blocks = (fused_recv_wave_items + waves - 1) / waves;
        // Every receive workgroup goes through the batch's entries for the own counts.  Small ones of four waves do better with
        // half as many of them once there are entries enough, as long as the send workgroups in front leave them places in
        // the first round.  Microseconds of a step, top-8 in fp8 unless said, 1024 of them / 512:
        //   580 x 4096   36.7 / 35.1    700 x 4096  42.2 / 40.8    820 x 4096  49.7 / 47.5    936 x 4096, top-6  44.6 / 43.1
        //   1000 x 4096  56.1 / 55.4    600 x 2048 bf16  30.3 / 29.7    900 x 2048 bf16  36.9 / 35.6    1500 x 4096, top-4  49.1 / 48.6
        //   400 x 4096   28.4 / 28.3    500 x 2048 bf16  23.8 / 24.6    1100 x 2048 bf16  44.7 / 45.6    2000 x 4096, top-4  58.9 / 60.0
        // Workgroups of eight waves: 340 x 7168 bf16 47.6 / 48.2, 1000 x 7168 93.3 / 94.0.  Where far more rows come in than the
        // batch sends, three launches against one with 512: 1000 of 2048, 14900 rows 23.5 / 15.3; 600 of 4096, 14500 33.2 / 24.1.
        const bool few = waves <= 4 && n > kFusedFewFrom && n <= kFusedMaxEntries && num_tokens <= kFusedFewTokens;
        const int64_t most = tokens_per_block > 1 || few ? 512 : 1024;
        fused_recv_blocks = fused_recv_blocks < 1 ? 1 : (fused_recv_blocks > most ? most : fused_recv_blocks);
        const int64_t total = int64_t(num_send_blocks) + 1 + fused_recv_blocks + 1;  // + counting, + metadata
        EP_HOST_ASSERT(total < (int64_t(1) << 31));
        const int num_segments = fused_recv->num_local_experts * fused_recv->num_ranks;
        const size_t need_recv = size_t(num_segments + 1 + fused_recv->num_local_experts) * sizeof(int32_t);
        const size_t need_count = size_t(num_experts) * sizeof(int32_t);
        const size_t lds = need_recv > need_count ? need_recv : need_count;
        const RecvArgs ra = *fused_recv;
        // Token rows read and K copies written by the send workgroups, staged rows read and packed rows
        // written by the receive workgroups.  From 64 MB on (about 350 tokens at hidden 7168, top-8) the
        // launch streams: at 512 to 1024 tokens that changes nothing when the caches are clean and takes
        // 11 to 16 % off when they are full of another call's dirty lines (44 against 50 us at 1024 tokens).
        const int64_t payload = row_payload_bytes(hidden, row_format);
        const int64_t fused_traffic = int64_t(num_tokens) * (int64_t(hidden) * 2 + int64_t(num_topk) * payload) +
                                      2 * (fused_recv_wave_items >> ra.parts_log2) * payload;
        const bool fused_streams = fused_traffic > send_stream_bytes();
#define DEEPEP_LAUNCH_FUSED_AS(FMT, STREAM, MANY)                                                                    \
    launch(ll_dispatch_fused_kernel<FMT, STREAM, MANY>, dim3(unsigned(total)), waves * kWave, lds, stream, sa, ra,    \
           blocks_per_token, num_send_blocks)
#define DEEPEP_LAUNCH_FUSED(FMT)                                                                                     \
    do {                                                                                                             \
        if (tokens_per_block > 1) {                                                                                  \
            if (fused_streams) DEEPEP_LAUNCH_FUSED_AS(FMT, true, true);                                              \
            else DEEPEP_LAUNCH_FUSED_AS(FMT, false, true);                                                           \
        } else {                                                                                                     \
            if (fused_streams) DEEPEP_LAUNCH_FUSED_AS(FMT, true, false);                                             \
            else DEEPEP_LAUNCH_FUSED_AS(FMT, false, false);                                                          \
        }                                                                                                            \
    } while (0)
        switch (row_format) {
            case kRowBF16: DEEPEP_LAUNCH_FUSED(kRowBF16); break;
            case kRowFP8: DEEPEP_LAUNCH_FUSED(kRowFP8); break;
            case kRowFP8Pow2: DEEPEP_LAUNCH_FUSED(kRowFP8Pow2); break;
            default: DEEPEP_LAUNCH_FUSED(kRowFP8UE8M0); break;
        }
#undef DEEPEP_LAUNCH_FUSED
#undef DEEPEP_LAUNCH_FUSED_AS
        EP_LAUNCH_CHECK();
        return 0;
    }

    // The receive index rides along with the rows of a ranked one-call dispatch, for whose own counts it reads all histograms
    FusedIndexArgs index = {};
    int index_rows = 0;
    if (fused_index != nullptr && ranked && !batch.first_in_finish) {
        index = *fused_index;
        index.chunk_hist = batch.hists, index.num_chunks = batch.num_chunks;
        index_rows = (num_experts + blocks_per_token - 1) / blocks_per_token;
        if (num_tokens + 1 + index_rows > 65535) index_rows = 0, index = FusedIndexArgs{};
    }
    if (index_was_fused != nullptr) *index_was_fused = index_rows > 0;
    const DirectOut direct = own_rows_direct != nullptr ? *own_rows_direct : DirectOut{nullptr, nullptr, nullptr};
    // rows read once and written K times (about that many: a dropped selection writes nothing)
    const int64_t traffic = int64_t(num_src) * num_tokens *
                            (int64_t(hidden) * 2 + int64_t(num_topk) * row_payload_bytes(hidden, row_format));
    const bool streams = traffic > send_stream_bytes();
    // + the index rows, + the counting row (ll_rank_finish_kernel has the counts)
    const dim3 grid(blocks_per_token, index_rows + token_blocks + (ranked && batch.in_full ? 0 : 1), num_src);
    if (grid.y == 0) return 0;
    const size_t lds = size_t(index_rows > 0 ? 2 * (num_experts + 1) : num_experts + 1) * sizeof(int32_t);
    int topk_log2 = 0;
    while ((1 << topk_log2) < num_topk) ++topk_log2;
#define DEEPEP_LAUNCH_SEND_AS(FMT, STREAM)                                                                             \
    do {                                                                                                               \
        if (ranked)                                                                                                    \
            launch(ll_send_ranked_kernel<FMT, STREAM>, grid, waves * kWave, lds, stream, sa, direct, batch, index,         \
                                                                                     index_rows, topk_log2);           \
        else if (tokens_per_block > 1)                                                                                 \
            launch(ll_send_kernel<FMT, STREAM, true>, grid, waves * kWave, lds, stream, sa);                           \
        else                                                                                                           \
            launch(ll_send_kernel<FMT, STREAM, false>, grid, waves * kWave, lds, stream, sa);                          \
    } while (0)
#define DEEPEP_LAUNCH_SEND(FMT)                            \
    do {                                                   \
        if (streams) DEEPEP_LAUNCH_SEND_AS(FMT, true);     \
        else DEEPEP_LAUNCH_SEND_AS(FMT, false);            \
    } while (0)
    switch (row_format) {
        case kRowBF16: DEEPEP_LAUNCH_SEND(kRowBF16); break;
        case kRowFP8: DEEPEP_LAUNCH_SEND(kRowFP8); break;
        case kRowFP8Pow2: DEEPEP_LAUNCH_SEND(kRowFP8Pow2); break;
        default: DEEPEP_LAUNCH_SEND(kRowFP8UE8M0); break;
    }
#undef DEEPEP_LAUNCH_SEND
#undef DEEPEP_LAUNCH_SEND_AS
    EP_LAUNCH_CHECK();
    return 0;
}

}  // namespace deepep

using namespace deepep;

extern "C" {

size_t deepep_ll_row_data_bytes(int hidden, int row_format) { return size_t(row_data_bytes(hidden, row_format)); }
size_t deepep_ll_row_scale_bytes(int hidden, int row_format) { return size_t(row_scale_bytes(hidden, row_format)); }
size_t deepep_ll_row_stride(int hidden, int row_format) { return size_t(row_stride_bytes(hidden, row_format)); }
size_t deepep_ll_row_payload_bytes(int hidden, int row_format) { return size_t(row_payload_bytes(hidden, row_format)); }

size_t deepep_ll_segment_workspace_bytes(int num_experts, int num_max_dispatch_tokens_per_rank) {
    return size_t(segment_workspace_bytes(num_experts, num_max_dispatch_tokens_per_rank));
}

size_t deepep_ll_dispatch_workspace_bytes(int num_tokens, int num_topk, int num_experts) {
    return size_t(route_scratch_bytes(num_tokens, num_topk, num_experts));
}

int deepep_ll_dispatch_send(const void* x, const int64_t* topk_idx, int num_tokens, int hidden, int num_topk,
                            int num_experts, int num_ranks, int rank, int num_max_dispatch_tokens_per_rank,
                            int row_format, void* recv_staging, int32_t* recv_count, void* send_slots,
                            int32_t* send_count, int32_t* pair_slot, void* workspace, size_t workspace_bytes,
                            void* stream) {
    clear_error();
    if (int rc = check_ll_shape(num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                                num_max_dispatch_tokens_per_rank, row_format))
        return rc;
    EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
    EP_HOST_ASSERT(recv_staging != nullptr && recv_count != nullptr);
    EP_HOST_ASSERT(send_count != nullptr && pair_slot != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(recv_staging) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_slots) & 15) == 0);
    return launch_send_side(x, topk_idx, nullptr, 1, num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                            num_max_dispatch_tokens_per_rank, row_format, recv_staging, recv_count, send_slots,
                            send_count, pair_slot, workspace, workspace_bytes,
                            reinterpret_cast<hipStream_t>(stream));
}

// Device address of `scratch` on the GPU that `stream` runs on, looked up once per device.
static int static_route_scratch(hipStream_t stream, void** out) {
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static void* address[kMaxDevices] = {};
    int device = -1;
    EP_HIP_CHECK(hipGetDevice(&device));
    EP_HOST_ASSERT(device >= 0 && device < kMaxDevices);
    if (stream != nullptr) {  // the symbol's address is per device: the stream must be the current device's
        int stream_device = -1;
        EP_HIP_CHECK(hipStreamGetDevice(stream, &stream_device));
        EP_HOST_ASSERT(stream_device == device);
    }
    std::lock_guard<std::mutex> lock(mutex);
    if (address[device] == nullptr) {
        void* p = nullptr;
        EP_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        EP_HOST_ASSERT(p != nullptr);
        address[device] = p;
    }
    *out = address[device];
    return 0;
}

int deepep_ll_dispatch_send_static(const void* x, const int64_t* topk_idx, int num_tokens, int hidden, int num_topk,
                                   int num_experts, int num_ranks, int rank, int num_max_dispatch_tokens_per_rank,
                                   int row_format, void* recv_staging, int32_t* recv_count, void* send_slots,
                                   int32_t* send_count, int32_t* pair_slot, void* stream) {
    clear_error();
    if (int rc = check_ll_shape(num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                                num_max_dispatch_tokens_per_rank, row_format))
        return rc;
    const size_t need = size_t(chunk_hist_bytes(num_tokens, num_topk, num_experts));
    if (need > kStaticScratchBytes) {
        set_error("Assertion", __FILE_NAME__, __LINE__,
                  "batch too large for the static route scratch: ceil(num_tokens / floor(2048 / num_topk)) * "
                  "num_experts * 4 bytes must not exceed 1 MiB; use deepep_ll_dispatch_send with a workspace");
        return 1;
    }
    void* route_scratch = nullptr;
    if (int rc = static_route_scratch(reinterpret_cast<hipStream_t>(stream), &route_scratch)) return rc;
    EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
    EP_HOST_ASSERT(recv_staging != nullptr && recv_count != nullptr);
    EP_HOST_ASSERT(send_count != nullptr && pair_slot != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(recv_staging) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_slots) & 15) == 0);
    return launch_send_side(x, topk_idx, nullptr, 1, num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                            num_max_dispatch_tokens_per_rank, row_format, recv_staging, recv_count, send_slots,
                            send_count, pair_slot, route_scratch, kStaticScratchBytes,
                            reinterpret_cast<hipStream_t>(stream));
}

int deepep_ll_dispatch_send_by_dest(const void* x, const int64_t* topk_idx, int num_tokens, int hidden, int num_topk,
                                    int num_experts, int num_ranks, int rank, int num_max_dispatch_tokens_per_rank,
                                    int row_format, void* send_rows, int64_t send_row_capacity, int32_t* send_count,
                                    int32_t* send_expert_prefix, int32_t* send_counts, int64_t* send_cumsum,
                                    int32_t* pair_slot, void* workspace, size_t workspace_bytes, void* stream) {
    clear_error();
    if (int rc = check_ll_shape(num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                                num_max_dispatch_tokens_per_rank, row_format))
        return rc;
    EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
    EP_HOST_ASSERT(send_count != nullptr && send_expert_prefix != nullptr && send_counts != nullptr &&
                   send_cumsum != nullptr && pair_slot != nullptr);
    // every live pair sends one row, and an expert takes at most M of them
    const int64_t most_rows = std::min<int64_t>(int64_t(num_tokens) * num_topk,
                                                int64_t(num_experts) * num_max_dispatch_tokens_per_rank);
    EP_HOST_ASSERT(send_row_capacity >= most_rows);
    EP_HOST_ASSERT(most_rows == 0 || send_rows != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_rows) & 15) == 0);
    const ByDestTables tables = {send_expert_prefix, send_counts, send_cumsum};
    return launch_send_side(x, topk_idx, nullptr, 1, num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                            num_max_dispatch_tokens_per_rank, row_format, nullptr, nullptr, send_rows, send_count,
                            pair_slot, workspace, workspace_bytes, reinterpret_cast<hipStream_t>(stream), nullptr, 0,
                            nullptr, &tables);
}

int deepep_loopback_dispatch_from_peers(const void* x, const int64_t* topk_idx, const int32_t* src_ranks,
                                        int num_src, int num_tokens, int hidden, int num_topk, int num_experts,
                                        int num_ranks, int rank, int num_max_dispatch_tokens_per_rank,
                                        int row_format, void* recv_staging, int32_t* recv_count, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    clear_error();
    if (int rc = check_ll_shape(num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                                num_max_dispatch_tokens_per_rank, row_format))
        return rc;
    EP_HOST_ASSERT(num_src >= 0 && num_src <= 65535);
    if (num_src == 0) return 0;
    EP_HOST_ASSERT(src_ranks != nullptr && recv_staging != nullptr && recv_count != nullptr);
    EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(recv_staging) & 15) == 0);
    return launch_send_side(x, topk_idx, src_ranks, num_src, num_tokens, hidden, num_topk, num_experts, num_ranks,
                            rank, num_max_dispatch_tokens_per_rank, row_format, recv_staging, recv_count, nullptr,
                            nullptr, nullptr, workspace, workspace_bytes, reinterpret_cast<hipStream_t>(stream));
}

static int check_recv_args(const void* recv_staging, const int32_t* recv_count, int hidden, int num_experts,
                           int num_ranks, int max_tokens, int row_format, void* packed_recv_x,
                           void* packed_recv_scales, int32_t* packed_recv_src_info, int64_t* packed_recv_layout_range,
                           int32_t* packed_recv_count) {
    EP_HOST_ASSERT(hidden > 0 && hidden % 128 == 0);
    EP_HOST_ASSERT(num_ranks > 0 && num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(max_tokens > 0);
    EP_HOST_ASSERT(row_format >= kRowBF16 && row_format <= kRowFP8UE8M0);
    EP_HOST_ASSERT(row_format != kRowFP8UE8M0 || (hidden / 128) % 4 == 0);
    EP_HOST_ASSERT(num_experts <= 1024);
    EP_HOST_ASSERT(recv_staging != nullptr && recv_count != nullptr && packed_recv_x != nullptr);
    EP_HOST_ASSERT(row_format == kRowBF16 || packed_recv_scales != nullptr);
    EP_HOST_ASSERT(packed_recv_src_info != nullptr && packed_recv_layout_range != nullptr &&
                   packed_recv_count != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(recv_staging) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(recv_count) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(packed_recv_x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(packed_recv_scales) & 3) == 0);
    EP_HOST_ASSERT(int64_t(num_experts) * max_tokens < (int64_t(1) << 31));
    return 0;
}

static RecvArgs make_recv_args(const void* recv_staging, const int32_t* recv_count, int hidden, int num_experts,
                               int num_ranks, int max_tokens, int row_format, void* packed_recv_x,
                               void* packed_recv_scales, int32_t* packed_recv_src_info,
                               int64_t* packed_recv_layout_range, int32_t* packed_recv_count, int32_t* stats,
                               int64_t expected_rows, const ObservedRows& observed) {
    RecvArgs ra;
    ra.recv_staging = reinterpret_cast<const uint8_t*>(recv_staging);
    ra.recv_count = recv_count;
    ra.hidden = hidden, ra.num_local_experts = num_experts / num_ranks, ra.num_ranks = num_ranks;
    ra.max_tokens = max_tokens, ra.fmt = row_format, ra.expert_of = make_rank_divider(num_ranks);
    const int64_t rows = estimated_rows(expected_rows, num_experts, max_tokens), row_bytes = row_data_bytes(hidden, row_format);
    ra.parts_log2 = choose_row_parts_log2(rows, row_bytes, num_experts);
    // A row of up to 4 KiB is what a wave loads at once (kRecvDepth): with enough rows to occupy the chip a wave
    // takes it whole, which halves the lookups and the trips of a wave.  The dispatch alone, halves against whole
    // rows: 1200 x 4096 bytes 7.4 -> 6.8 us, 2400 x 4096 12.0 -> 10.7, 4072 x 4096 17.0 -> 15.8, 2048 x 2048 8.7 ->
    // 8.0; 1024 x 4096 6.8 both ways; rows of 7168 bytes lose (40.9 -> 43.2), and so does the combine's row return.
    if (rows > 1024 && row_bytes <= int64_t(kRecvDepth) * kWave * 16) ra.parts_log2 = 0;
    ra.packed_x = reinterpret_cast<uint8_t*>(packed_recv_x);
    ra.packed_scales = reinterpret_cast<uint8_t*>(packed_recv_scales);
    ra.src_info = packed_recv_src_info, ra.layout_range = packed_recv_layout_range;
    ra.packed_count = packed_recv_count, ra.stats = stats;
    ra.observed = observed;
    return ra;
}

// own_rank >= 0: the send kernel, which has finished, put this rank's own rows at their packed
// position and their counts into recv_count; they are not copied again.
static int launch_recv_side(const void* recv_staging, const int32_t* recv_count, int hidden, int num_experts,
                            int num_ranks, int num_max_dispatch_tokens_per_rank, int row_format,
                            void* packed_recv_x, void* packed_recv_scales, int32_t* packed_recv_src_info,
                            int64_t* packed_recv_layout_range, int32_t* packed_recv_count,
                            int32_t* cumulative_local_expert_recv_stats, int64_t expected_rows, void* workspace,
                            size_t workspace_bytes, int own_rank, void* stream, bool index_done = false,
                            const ObservedRows& observed = ObservedRows{nullptr, 0}) {
    if (int rc = check_recv_args(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                 num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                 packed_recv_src_info, packed_recv_layout_range, packed_recv_count))
        return rc;
    const int num_local_experts = num_experts / num_ranks;
    const int64_t max_rows = int64_t(num_experts) * num_max_dispatch_tokens_per_rank;
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    const bool large = estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank) > kLargeBatchRows;
    if (large && workspace != nullptr) {
        EP_HOST_ASSERT(workspace_bytes >= size_t(segment_workspace_bytes(num_experts, num_max_dispatch_tokens_per_rank)));
        EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(workspace) & 15) == 0);
        int32_t* flat = reinterpret_cast<int32_t*>(workspace);
        RowDesc* desc = reinterpret_cast<RowDesc*>(reinterpret_cast<uint8_t*>(workspace) +
                                                   (((int64_t(num_experts) + 1) * 4 + 255) & ~int64_t(255)));
        if (!index_done) {  // (a large one-call dispatch builds the index inside its send launch)
            launch(ll_segment_index_kernel, num_experts, kIndexThreads, 0, hs,
                recv_count, num_local_experts, num_ranks, own_rank, num_max_dispatch_tokens_per_rank,
                packed_recv_layout_range, packed_recv_count, cumulative_local_expert_recv_stats, flat, desc, observed);
            EP_LAUNCH_CHECK();
        }
        const int64_t data_bytes = row_data_bytes(hidden, row_format);
        const int64_t scale_bytes = row_scale_bytes(hidden, row_format);
        const int num_vec = int(data_bytes / 16);
        FlatTails tails;
        tails.scale_dst = reinterpret_cast<uint8_t*>(packed_recv_scales), tails.src_info = packed_recv_src_info;
        tails.scale_dwords = packed_recv_scales != nullptr ? uint32_t(scale_bytes / 4) : 0u;
        tails.scale_off = uint32_t(align16(data_bytes));
        tails.info_off = uint32_t(align16(data_bytes) + align16(scale_bytes));
        // rows that are in place already are not described: of a balanced batch, one in num_ranks
        const int64_t rows = estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank);
        launch_rows_flat(flat + num_experts, desc, max_rows, own_rank >= 0 ? rows - rows / num_ranks : rows, recv_staging,
                         row_stride_bytes(hidden, row_format), num_vec, packed_recv_x, nullptr, data_bytes, &tails, hs);
        EP_LAUNCH_CHECK();
        return 0;
    }
    const RecvArgs ra = make_recv_args(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                       num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                       packed_recv_src_info, packed_recv_layout_range, packed_recv_count,
                                       cumulative_local_expert_recv_stats, expected_rows, observed);
    int64_t blocks = ((max_rows << ra.parts_log2) + 3) / 4;
    const int64_t cap = large ? 4096 : 1024;
    if (blocks > cap) blocks = cap;
    const size_t lds = size_t(num_experts + 1 + num_local_experts) * sizeof(int32_t);
    launch(ll_recv_kernel, dim3(unsigned(blocks) + 1), 256, lds, hs, ra, own_rank);  // + the metadata workgroup
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_ll_dispatch_recv(const void* recv_staging, const int32_t* recv_count, int hidden, int num_experts,
                            int num_ranks, int num_max_dispatch_tokens_per_rank, int row_format,
                            void* packed_recv_x, void* packed_recv_scales, int32_t* packed_recv_src_info,
                            int64_t* packed_recv_layout_range, int32_t* packed_recv_count,
                            int32_t* cumulative_local_expert_recv_stats, int64_t expected_rows, void* workspace,
                            size_t workspace_bytes, void* stream) {
    clear_error();
    return launch_recv_side(recv_staging, recv_count, hidden, num_experts, num_ranks,
                            num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                            packed_recv_src_info, packed_recv_layout_range, packed_recv_count,
                            cumulative_local_expert_recv_stats, expected_rows, workspace, workspace_bytes, -1, stream);
}

int deepep_ll_dispatch_is_single_launch(int num_tokens, int num_topk, int num_experts,
                                        int num_max_dispatch_tokens_per_rank, int64_t expected_rows) {
    return int64_t(num_tokens) * num_topk <= kFusedMaxEntries &&
                   estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank) <= kLargeBatchRows
               ? 1
               : 0;
}

int deepep_ll_dispatch_takes_one_launch(int num_tokens, int hidden, int num_topk, int num_experts,
                                        int num_max_dispatch_tokens_per_rank, int row_format, int64_t expected_rows) {
    return dispatch_in_one_launch(num_tokens, num_topk, num_experts, num_max_dispatch_tokens_per_rank, hidden, row_format,
                                  expected_rows)
               ? 1
               : 0;
}

int deepep_ll_dispatch_observed(const void* x, const int64_t* topk_idx, int num_tokens, int hidden, int num_topk,
                                int num_experts, int num_ranks, int rank, int num_max_dispatch_tokens_per_rank, int row_format,
                                void* recv_staging, int32_t* recv_count, void* send_slots, int32_t* send_count,
                                int32_t* pair_slot, void* packed_recv_x, void* packed_recv_scales,
                                int32_t* packed_recv_src_info, int64_t* packed_recv_layout_range, int32_t* packed_recv_count,
                                int32_t* cumulative_local_expert_recv_stats, int64_t expected_rows, void* workspace,
                                size_t workspace_bytes, void* segment_workspace, size_t segment_workspace_bytes,
                                uint64_t* observed_host, void* stream) {
    clear_error();
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(observed_host) & 7) == 0);
    const ObservedRows observed = {observed_host, uint32_t(num_tokens < 0 ? 0 : num_tokens)};
    const int64_t max_rows = int64_t(num_experts) * num_max_dispatch_tokens_per_rank;
    if (int rc = check_ll_shape(num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                                num_max_dispatch_tokens_per_rank, row_format))
        return rc;
    const bool fused = dispatch_in_one_launch(num_tokens, num_topk, num_experts, num_max_dispatch_tokens_per_rank, hidden,
                                              row_format, expected_rows);
    const bool large = segment_workspace != nullptr && num_experts <= 1024 &&
                       estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank) > kLargeBatchRows;
    if (large) {
        EP_HOST_ASSERT(segment_workspace_bytes >=
                       size_t(deepep::segment_workspace_bytes(num_experts, num_max_dispatch_tokens_per_rank)));
        EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(segment_workspace) & 15) == 0);
    }
    if (!fused) {
        // The two phases back to back, with the single launch's shortcut: the send side writes the
        // rows for this rank's own experts straight to their packed position behind the lower ranks'
        // rows (whose counts are in recv_count already), and the receive side copies the rest.
        EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
        EP_HOST_ASSERT(recv_staging != nullptr && recv_count != nullptr && pair_slot != nullptr && send_count != nullptr);
        EP_HOST_ASSERT(workspace != nullptr);
        EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
        EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_slots) & 15) == 0);
        if (int rc = check_recv_args(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                     num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                     packed_recv_src_info, packed_recv_layout_range, packed_recv_count))
            return rc;
        const DirectOut direct = {reinterpret_cast<uint8_t*>(packed_recv_x),
                                  reinterpret_cast<uint8_t*>(packed_recv_scales), packed_recv_src_info};
        // When the receive side will run as index + flat copy, the index is built by extra workgroups of
        // the send launch: three launches (slots, send + index, copy) instead of four.
        FusedIndexArgs index = {};
        if (large) {
            index.recv_count = recv_count;
            index.num_experts = num_experts, index.num_local_experts = num_experts / num_ranks;
            index.num_ranks = num_ranks, index.rank = rank, index.max_tokens = num_max_dispatch_tokens_per_rank;
            index.layout_out = packed_recv_layout_range, index.packed_count = packed_recv_count;
            index.stats = cumulative_local_expert_recv_stats;
            index.observed = observed;
            index.flat_out = reinterpret_cast<int32_t*>(segment_workspace);
            index.desc = reinterpret_cast<RowDesc*>(reinterpret_cast<uint8_t*>(segment_workspace) +
                                                    (((int64_t(num_experts) + 1) * 4 + 255) & ~int64_t(255)));
        }
        bool index_done = false;
        if (int rc = launch_send_side(x, topk_idx, nullptr, 1, num_tokens, hidden, num_topk, num_experts, num_ranks,
                                      rank, num_max_dispatch_tokens_per_rank, row_format, recv_staging, recv_count,
                                      send_slots, send_count, pair_slot, workspace, workspace_bytes,
                                      reinterpret_cast<hipStream_t>(stream), nullptr, 0, &direct, nullptr,
                                      large ? &index : nullptr, &index_done))
            return rc;
        return launch_recv_side(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                packed_recv_src_info, packed_recv_layout_range, packed_recv_count,
                                cumulative_local_expert_recv_stats, expected_rows, segment_workspace,
                                segment_workspace_bytes, rank, stream, index_done, observed);
    }
    EP_HOST_ASSERT(num_tokens == 0 || (x != nullptr && topk_idx != nullptr));
    EP_HOST_ASSERT(send_count != nullptr && pair_slot != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_slots) & 15) == 0);
    if (int rc = check_recv_args(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                 num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                 packed_recv_src_info, packed_recv_layout_range, packed_recv_count))
        return rc;
    const RecvArgs ra = make_recv_args(recv_staging, recv_count, hidden, num_experts, num_ranks,
                                       num_max_dispatch_tokens_per_rank, row_format, packed_recv_x, packed_recv_scales,
                                       packed_recv_src_info, packed_recv_layout_range, packed_recv_count,
                                       cumulative_local_expert_recv_stats, expected_rows, observed);
    int64_t rows = expected_rows > 0 ? expected_rows : int64_t(num_max_dispatch_tokens_per_rank) * num_topk;
    rows += rows / 8 + 16;
    if (rows > max_rows) rows = max_rows;
    return launch_send_side(x, topk_idx, nullptr, 1, num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
                            num_max_dispatch_tokens_per_rank, row_format, recv_staging, recv_count, send_slots,
                            send_count, pair_slot, workspace, workspace_bytes,
                            reinterpret_cast<hipStream_t>(stream), &ra, rows << ra.parts_log2);
}

// Kernels and grids are chosen by it, never results.  The rows come from the other ranks, so they do not grow with
// this rank's own tokens: scaled up, 1 token that received 2100 rows made 4 tokens expect 8400 and leave the single
// launch (a step of 4 tokens 18.8 -> 27.8 us).  They are scaled down, because the ranks leave a prefill together: a
// decode step of 128 tokens sized by the 32768 rows of one took 35.0 us instead of 18.8.  A hint that is too small
// costs a looping copy (1000 tokens, 165885 rows: 1550 us sized for 8000, 1199 for what arrives).
int64_t deepep_ll_expected_rows(int num_tokens, int num_topk, int num_experts, int num_max_dispatch_tokens_per_rank,
                                uint64_t observed) {
    const int64_t balanced = std::max<int64_t>(num_tokens, 1) * num_topk;
    const int64_t tokens = int64_t(observed >> 32), rows = int64_t(observed & 0xffffffffu);
    if (tokens == 0) return balanced;
    const int64_t again = num_tokens < tokens ? rows * num_tokens / tokens : rows;
    return std::max(balanced, std::min(again, int64_t(num_experts) * num_max_dispatch_tokens_per_rank));
}

// Layers that share a buffer report in turn.  Sized by the last word alone, a hot layer (166336 rows, 64 ranks, 1000
// tokens of hidden 7168) and a cold one (7959) in turn size each other: 1384 + 384 us a step where their own hints give
// 1140 + 101.  The geometric mean of the two: 1198 + 160; nearer to either, 1159 + 228 and 1264 + 121.
int64_t deepep_ll_expected_rows_of_two(int num_tokens, int num_topk, int num_experts,
                                       int num_max_dispatch_tokens_per_rank, uint64_t observed_a, uint64_t observed_b) {
    const int64_t tokens_a = int64_t(observed_a >> 32), tokens_b = int64_t(observed_b >> 32);
    if (tokens_b == 0 || (tokens_a >= num_tokens && tokens_b < num_tokens)) observed_b = observed_a;
    else if (tokens_a == 0 || (tokens_b >= num_tokens && tokens_a < num_tokens)) observed_a = observed_b;
    const int64_t a = deepep_ll_expected_rows(num_tokens, num_topk, num_experts, num_max_dispatch_tokens_per_rank, observed_a);
    const int64_t b = deepep_ll_expected_rows(num_tokens, num_topk, num_experts, num_max_dispatch_tokens_per_rank, observed_b);
    return a == b ? a : int64_t(std::sqrt(double(a) * double(b)));
}

int deepep_ll_dispatch(const void* x, const int64_t* topk_idx, int num_tokens, int hidden, int num_topk,
                       int num_experts, int num_ranks, int rank, int num_max_dispatch_tokens_per_rank, int row_format,
                       void* recv_staging, int32_t* recv_count, void* send_slots, int32_t* send_count,
                       int32_t* pair_slot, void* packed_recv_x, void* packed_recv_scales,
                       int32_t* packed_recv_src_info, int64_t* packed_recv_layout_range, int32_t* packed_recv_count,
                       int32_t* cumulative_local_expert_recv_stats, int64_t expected_rows, void* workspace,
                       size_t workspace_bytes, void* segment_workspace, size_t segment_workspace_bytes,
                       void* stream) {
    return deepep_ll_dispatch_observed(
        x, topk_idx, num_tokens, hidden, num_topk, num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank,
        row_format, recv_staging, recv_count, send_slots, send_count, pair_slot, packed_recv_x, packed_recv_scales,
        packed_recv_src_info, packed_recv_layout_range, packed_recv_count, cumulative_local_expert_recv_stats,
        expected_rows, workspace, workspace_bytes, segment_workspace, segment_workspace_bytes, nullptr, stream);
}

}  // extern "C"
