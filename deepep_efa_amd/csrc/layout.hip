// Route counting and layout for the normal-mode path: per-expert / per-rank
// counts with the token x rank membership matrix, the per-rank token sort,
// the channel prefix matrix, and the row gather that packs per-rank send
// buffers.
#include "common.hpp"
#include "../../include/deepep_hip.h"

#include <algorithm>

namespace deepep {

constexpr int kLayoutThreads = 256;
constexpr int kMaxRankWords = 4;  // membership bitmask: up to 256 ranks
constexpr int kLayoutOneBlockThreads = 1024;
// Up to here one workgroup counts everything and no second launch adds up partial rows: one or two tokens a thread.
// Microseconds of the one launch against the two, in a row (the second also takes the host 2.3):
//   ranks        8            16           32            64
//   400 tokens   2.9 / 4.1    3.3 / 4.4    3.8 / 4.8     4.8 / 5.4
//   700          3.0 / 4.1    3.4 / 4.4    3.9 / 4.8     4.8 / 5.5
//   1024         3.3 / 4.3    3.7 / 4.5    4.2 / 4.8     5.9 / 5.5
//   1500         4.3 / 4.3    5.0 / 4.6    6.0 / 4.9    10.3 / 5.5
//   2048         4.4 / 4.5    5.3 / 4.8    6.4 / 5.1    11.4 / 5.9
//   3000         5.6 / 4.7    6.8 / 4.9    8.5 / 5.2    16.6 / 6.0
// Past 1024 tokens up to 16384 entries, which one workgroup takes one after another (8 ranks, 2048 tokens, top-8 4.9 / 5.0, top-12
// 5.7 / 5.3, top-16 10.4 / 6.8, top-32 17.9 / 8.5), and past 512 with more than 32 ranks only of whole eights, whose bytes are stored a
// word at a time (63 ranks, 768 tokens 9.2 / 7.1; 250 ranks, 700 tokens 27.1 / 16.1).
inline int layout_one_block_tokens(int num_ranks, int num_topk) {
    if (num_ranks <= 8) return std::min(2048, std::max(1024, 16384 / num_topk));
    return num_ranks <= 32 ? 1024 : num_ranks % 8 == 0 ? 768 : 512;
}

// Spreads the 8 bits of b into 8 bytes (byte i = bit i, value 0 or 1).
__device__ __forceinline__ uint64_t bits_to_bool_bytes(uint32_t b) {
    uint64_t x = (uint64_t(b & 0xffu) * 0x0101010101010101ull) & 0x8040201008040201ull;
    return ((x + 0x7f7f7f7f7f7f7f7full) >> 7) & 0x0101010101010101ull;
}

// 1 in every byte of v that is not zero.
__device__ __forceinline__ uint64_t nonzero_bytes(uint64_t v) {
    v |= v >> 4, v |= v >> 2, v |= v >> 1;
    return v & 0x0101010101010101ull;
}

// Sums over the wave of the eight bytes of v, which are 0 or 1, in its lanes first to first + 7: lane first + i gets byte i's;
// the others get what they hand in.  Four bytes are added up by one sum over the lanes, no byte past 64.
__device__ __forceinline__ int byte_sums_to_lanes(uint64_t v, int first, int otherwise) {
    const uint32_t lo = __builtin_amdgcn_readlane(wave_inclusive_sum(int(uint32_t(v))), kWave - 1);
    const uint32_t hi = __builtin_amdgcn_readlane(wave_inclusive_sum(int(uint32_t(v >> 32))), kWave - 1);
    const int i = lane_id() - first;
    return i >= 0 && i < 8 ? int((((i & 4) != 0 ? hi : lo) >> ((i & 3) * 8)) & 0xff) : otherwise;
}

// e / E_l by multiply-high (exact below 2^16 experts); magic 0 stands for E_l == 1.
__device__ __forceinline__ int rank_of_expert(uint32_t e, uint32_t rank_magic) {
    return rank_magic != 0 ? int(__umulhi(e, rank_magic)) : int(e);
}

// Counts the expert that entry 0 or 1 of two names and marks its rank, one of up to 64.
__device__ __forceinline__ void count_entry(u32x4 two, int which, int num_experts, uint32_t rank_magic, int32_t* hist,
                                            uint64_t& member) {
    const uint32_t e = two[which * 2];
    if (two[which * 2 + 1] != 0u || e >= uint32_t(num_experts)) return;
    atomicAdd(&hist[e], 1);
    member |= uint64_t(1) << (rank_of_expert(e, rank_magic) & 63);
}

// ---------------------------------------------------------------------
// get_dispatch_layout: one pass over topk_idx, one token per lane.
//   * per-expert pair counts: LDS histogram (integer adds — the result does
//     not depend on their order);
//   * per-rank and per-node distinct-token counts: each lane folds its K
//     selections into a rank bitmask, whose bits, spread to bytes, are added up
//     over the wave, four ranks at a time (a ballot and a popcount for each
//     rank: 64 tokens to 32 ranks 4.4 us, 1000 6.9);
//   * is_token_in_rank: the same bytes, 8 per store.
// Each workgroup writes a partial row [E | R | R/8]; with one workgroup the
// partial row is the result, otherwise a second small kernel adds the rows.
// What bounds it is latency, launches and, in one workgroup, instructions, not the
// few hundred KB it reads: hence one workgroup while that costs less than the
// second launch, and a bitmask of
// as many words as there are ranks for (an index into a longer one that the
// compiler cannot resolve goes through selects).
// Reference: csrc/kernels/layout.cu:9-121 (which re-reads topk_idx once per
// 4 experts / 8 ranks).
// ---------------------------------------------------------------------
template <int kRankWords>
__global__ __launch_bounds__(kLayoutOneBlockThreads) void layout_count_kernel(
    const int64_t* __restrict__ topk_idx, int num_tokens, int num_topk, int num_ranks, int num_experts,
    uint32_t rank_magic, int num_nodes, uint8_t* __restrict__ is_token_in_rank, int32_t* __restrict__ partial,
    int32_t* __restrict__ per_rank, int32_t* __restrict__ per_node, int32_t* __restrict__ per_expert) {
    extern __shared__ int32_t hist[];  // [E + R + nodes]
    const int tid = threadIdx.x, lane = lane_id(), threads = block_threads();
    const int width = num_experts + num_ranks + num_nodes;
    for (int j = tid; j < width; j += threads) hist[j] = 0;
    lds_barrier();

    // whole waves go round together: the sums below want every lane
    for (int t0 = blockIdx.x * threads; t0 < num_tokens; t0 += int(gridDim.x) * threads) {
        const int t = t0 + tid;
        uint64_t member[kRankWords];
#pragma unroll
        for (int q = 0; q < kRankWords; ++q) member[q] = 0;
        // The round's rows as one buffer: 16-byte loads, two entries each, that need no more than four-byte alignment, and
        // zeros past the last token.  (Entries one at a time: 1000 tokens 4.1 us, a line of cache a lane and load.)
        const int tokens = num_tokens - t0 < threads ? num_tokens - t0 : threads;
        const auto rows = row_buffer(reinterpret_cast<const uint8_t*>(topk_idx + int64_t(t0) * num_topk), tokens * num_topk * 8);
        for (int k0 = 0; k0 < num_topk; k0 += 8) {
            u32x4 two[4];  // all in flight before the first is used
            const auto load = [&](int u) { two[u] = load_row_u32x4<false>(rows, (tid * num_topk + k0 + 2 * u) * 8); };
            if constexpr (kRankWords == 1) {
                if (k0 + 8 <= num_topk) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) load(u);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (t < num_tokens) count_entry(two[u / 2], u % 2, num_experts, rank_magic, hist, member[0]);
                } else {  // no more loads and tests than there are entries: 8 ranks, 1024 tokens, top-2 3.2 -> 2.9 us
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (k0 + 2 * u >= num_topk) break;
                        load(u);
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        if (k0 + u >= num_topk) break;
                        if (t < num_tokens) count_entry(two[u / 2], u % 2, num_experts, rank_magic, hist, member[0]);
                    }
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) load(u);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t e = two[u / 2][u % 2 * 2];
                    if (two[u / 2][u % 2 * 2 + 1] != 0u || e >= uint32_t(num_experts) || k0 + u >= num_topk || t >= num_tokens) continue;
                    atomicAdd(&hist[e], 1);
                    const int r = rank_of_expert(e, rank_magic);
#pragma unroll
                    for (int q = 0; q < kRankWords; ++q)
                        if ((r >> 6) == q) member[q] |= uint64_t(1) << (r & 63);
                }
            }
        }
        // lane r keeps rank (q * 64 + r)'s count of the wave, so that one atomic per lane adds them all
        uint8_t* out = is_token_in_rank + int64_t(t) * num_ranks;
        const bool in_words = (num_ranks & 7) == 0;
#pragma unroll
        for (int q = 0; q < kRankWords; ++q) {
            const int begin = q * kWave, end = num_ranks < begin + kWave ? num_ranks : begin + kWave;
            int count = 0;
            if (!in_words && t < num_tokens)
                for (int r = begin; r < end; ++r) out[r] = uint8_t((member[q] >> (r - begin)) & 1);
            for (int r8 = begin; r8 < end; r8 += 8) {
                const uint64_t in = bits_to_bool_bytes(uint32_t(member[q] >> (r8 - begin)));
                count = byte_sums_to_lanes(in, r8 - begin, count);
                if (in_words && t < num_tokens) *reinterpret_cast<uint64_t*>(out + r8) = in;
            }
            if (count != 0) atomicAdd(&hist[num_experts + begin + lane], count);
            if (q * 8 < num_nodes) {  // 8 ranks per node (reference: NUM_MAX_NVL_PEERS, csrc/kernels/configs.cuh:3)
                const int in_node = byte_sums_to_lanes(nonzero_bytes(member[q]), 0, 0);
                if (in_node != 0) atomicAdd(&hist[num_experts + num_ranks + q * 8 + lane], in_node);
            }
        }
    }
    lds_barrier();
    if (gridDim.x == 1) {  // the partial row is the result
        for (int j = tid; j < width; j += threads) {
            if (j < num_experts)
                per_expert[j] = hist[j];
            else if (j < num_experts + num_ranks)
                per_rank[j - num_experts] = hist[j];
            else
                per_node[j - num_experts - num_ranks] = hist[j];
        }
        return;
    }
    int32_t* dst = partial + int64_t(blockIdx.x) * width;
    for (int j = tid; j < width; j += threads) dst[j] = hist[j];
}

__global__ __launch_bounds__(kLayoutThreads) void layout_reduce_kernel(const int32_t* __restrict__ partial,
                                                                       int num_partials, int num_experts,
                                                                       int num_ranks, int num_nodes,
                                                                       int32_t* __restrict__ per_rank,
                                                                       int32_t* __restrict__ per_node,
                                                                       int32_t* __restrict__ per_expert) {
    const int width = num_experts + num_ranks + num_nodes;
    const int j = blockIdx.x * kLayoutThreads + threadIdx.x;
    if (j >= width) return;
    int sum = 0;
    for (int p0 = 0; p0 < num_partials; p0 += 8) {  // eight loads in flight
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p0 + u < num_partials ? partial[int64_t(p0 + u) * width + j] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += v[u];
    }
    if (j < num_experts)
        per_expert[j] = sum;
    else if (j < num_experts + num_ranks)
        per_rank[j - num_experts] = sum;
    else
        per_node[j - num_experts - num_ranks] = sum;
}

// Tells a host that polls `report` that this workgroup of a routing sort is done (null: nobody asked): one word a
// workgroup, stored when everything the workgroup wrote is in memory that every stream, copy engine and the host see.
// So a host that has seen all words may use the results from another stream too, as after a wait for this one.  (Told
// the total as soon as it is known, the host is 2 to 3 us further ahead -- 131, 4096 and 12289 tokens through the whole
// dispatch side 38.5, 130.4, 412.5 us against 40.7, 132.5, 415.5 -- and a reader on another stream gets what the list
// held before.)  The whole workgroup takes part; `value` is thread 0's.
__device__ __forceinline__ void report_done(int64_t* report, int64_t value) {
    if (report == nullptr) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores have reached the XCD's L2
    __syncthreads();
    if (threadIdx.x == 0)  // the release writes that L2 back
        __hip_atomic_store(report + blockIdx.x, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------
// moe_routing_sort: stable partition of token ids by destination rank.
//   count:   per 1024-token chunk and rank, tokens bound for that rank
//            (ballot + popcount per wave, summed over the chunk's 16 waves);
//   scan:    one workgroup turns the [chunk][rank] table into write offsets
//            (rank-major, chunk-minor) and emits send_counts / send_cumsum;
//   scatter: the count pass again, this time writing the ids.
// Ascending token order inside a rank follows from the chunk/wave/lane order.
// Reference: csrc/kernels/efa_kernels.cu:220-318 (one thread per rank there).
// Small batches take the one-launch variant further down.
// ---------------------------------------------------------------------
constexpr int kSortChunk = 1024;

template <bool kScatter>
__global__ __launch_bounds__(kSortChunk) void routing_sort_pass_kernel(
    const uint8_t* __restrict__ is_token_in_rank, int num_tokens, int num_ranks, int32_t* __restrict__ chunk_table,
    int64_t* __restrict__ sorted_token_ids, int32_t* __restrict__ row_of_pair, const int64_t* __restrict__ total,
    int64_t* __restrict__ report) {
    extern __shared__ int32_t wave_cnt[];  // [16][R]
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block();
    const int c = blockIdx.x;
    const int t = c * kSortChunk + tid;
    const uint8_t* row = is_token_in_rank + int64_t(t) * num_ranks;
    for (int r = 0; r < num_ranks; ++r) {
        const bool in = t < num_tokens && row[r] != 0;
        const uint64_t votes = __ballot(in);
        if (lane == 0) wave_cnt[w * num_ranks + r] = __popcll(votes);
    }
    __syncthreads();
    if constexpr (!kScatter) {
        for (int r = tid; r < num_ranks; r += kSortChunk) {
            int sum = 0;
            for (int w2 = 0; w2 < kSortChunk / kWave; ++w2) sum += wave_cnt[w2 * num_ranks + r];
            chunk_table[int64_t(c) * num_ranks + r] = sum;
        }
    } else {
        // one thread per rank turns the 16 per-wave counts into the waves' first positions
        for (int r = tid; r < num_ranks; r += kSortChunk) {
            int run = chunk_table[int64_t(c) * num_ranks + r];
#pragma unroll
            for (int w2 = 0; w2 < kSortChunk / kWave; ++w2) {
                const int cnt = wave_cnt[w2 * num_ranks + r];
                wave_cnt[w2 * num_ranks + r] = run;
                run += cnt;
            }
        }
        __syncthreads();
        for (int r = 0; r < num_ranks; ++r) {
            const bool in = t < num_tokens && row[r] != 0;
            const uint64_t votes = __ballot(in);
            const int pos = wave_cnt[w * num_ranks + r] + __popcll(votes & lanes_below(lane));
            if (in) sorted_token_ids[pos] = t;
            if (row_of_pair != nullptr && t < num_tokens) row_of_pair[int64_t(t) * num_ranks + r] = in ? pos : -1;
        }
        report_done(report, report != nullptr ? *total : 0);
    }
}

__global__ __launch_bounds__(256) void routing_sort_scan_kernel(int32_t* __restrict__ chunk_table, int num_chunks,
                                                                int num_ranks, int32_t* __restrict__ send_counts,
                                                                int64_t* __restrict__ send_cumsum,
                                                                int64_t* __restrict__ report) {
    extern __shared__ int64_t rank_base[];  // [R + 1]
    const int tid = threadIdx.x;
    for (int r = tid; r < num_ranks; r += 256) {
        int sum = 0;
        for (int c = 0; c < num_chunks; ++c) sum += chunk_table[int64_t(c) * num_ranks + r];
        send_counts[r] = sum;
        rank_base[r + 1] = sum;
    }
    __syncthreads();
    if (tid == 0) {
        rank_base[0] = 0;
        for (int r = 0; r < num_ranks; ++r) rank_base[r + 1] += rank_base[r];
    }
    __syncthreads();
    for (int r = tid; r <= num_ranks; r += 256) send_cumsum[r] = rank_base[r];
    for (int r = tid; r < num_ranks; r += 256) {
        int run = int(rank_base[r]);
        for (int c = 0; c < num_chunks; ++c) {
            const int cnt = chunk_table[int64_t(c) * num_ranks + r];
            chunk_table[int64_t(c) * num_ranks + r] = run;
            run += cnt;
        }
    }
    report_done(report, rank_base[num_ranks]);
}

// ---------------------------------------------------------------------
// The same sort in one launch, for up to 8192 tokens and 64 ranks: one workgroup per destination
// rank, each thread a run of consecutive tokens.  The workgroup reads the whole membership matrix
// (a few tens of KiB, from L2), so besides the positions of its own rank's tokens (a scan of one
// count per thread) it gets the number of memberships of all lower ranks — where its ids start —
// from the same data, without waiting for anybody.  One barrier; 10 us of three launches become 4.
// ---------------------------------------------------------------------
constexpr int kSingleSortTokensPerThread = 8;
// Up to here 256 threads do it: the others' waves would issue the same instructions for no tokens, sixteen waves' worth
// on one compute unit.  256 against 1024 threads: 131 tokens, 16 ranks 2.8 / 3.2 us, 512 tokens, 8 ranks 2.9 / 3.15,
// 400 tokens, 16 ranks 3.2 / 3.3, 800 tokens, 32 ranks 5.1 / 3.9.
constexpr int kSmallSortTokens = 512;

// Bit r of the result = is_token_in_rank[t][r] != 0, for up to 64 ranks.
__device__ __forceinline__ uint64_t membership_mask(const uint8_t* row, int num_ranks) {
    uint64_t mask = 0;
    if ((num_ranks & 7) == 0 && (reinterpret_cast<uintptr_t>(row) & 7) == 0) {
        for (int r8 = 0; r8 < num_ranks; r8 += 8) {
            uint64_t v = *reinterpret_cast<const uint64_t*>(row + r8);
            v |= v >> 4, v |= v >> 2, v |= v >> 1;  // any bit of a byte -> its bit 0
            v &= 0x0101010101010101ull;
            mask |= ((v * 0x0102040810204080ull) >> 56) << r8;  // gather the eight bit-0s into one byte
        }
    } else {
        for (int r = 0; r < num_ranks; ++r) mask |= uint64_t(row[r] != 0) << r;
    }
    return mask;
}

template <int kThreads>
__global__ __launch_bounds__(kThreads) void routing_sort_single_kernel(
    const uint8_t* __restrict__ is_token_in_rank, int num_tokens, int num_ranks, int tokens_per_thread,
    int32_t* __restrict__ send_counts, int64_t* __restrict__ send_cumsum, int64_t* __restrict__ sorted_token_ids,
    int32_t* __restrict__ row_of_pair, int64_t* __restrict__ report) {
    constexpr int kWaves = kThreads / kWave;
    __shared__ int32_t wave_own[kWaves];    // tokens of this rank in each wave
    __shared__ int32_t wave_lower[kWaves];  // memberships of lower ranks in each wave
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block();
    const int r = blockIdx.x;
    const uint64_t lower_mask = (uint64_t(1) << r) - 1;
    const int first = tid * tokens_per_thread;
    uint32_t own_bits = 0;  // bit i: token first + i goes to rank r
    int lower = 0;
#pragma unroll
    for (int i = 0; i < kSingleSortTokensPerThread; ++i) {
        const int t = first + i;
        if (i < tokens_per_thread && t < num_tokens) {
            const uint64_t m = membership_mask(is_token_in_rank + int64_t(t) * num_ranks, num_ranks);
            own_bits |= uint32_t((m >> r) & 1) << i;
            lower += __popcll(m & lower_mask);
        }
    }
    const int own = __popc(own_bits);
    const int incl = wave_inclusive_sum(own);
    const int lower_wave = wave_inclusive_sum(lower);
    if (lane == kWave - 1) wave_own[w] = incl, wave_lower[w] = lower_wave;
    lds_barrier();
    int before = 0, total = 0, base = 0;
#pragma unroll
    for (int w2 = 0; w2 < kWaves; ++w2) {
        const int c = wave_own[w2];
        if (w2 < w) before += c;
        total += c;
        base += wave_lower[w2];
    }
    int64_t pos = int64_t(base) + before + incl - own;
#pragma unroll
    for (int i = 0; i < kSingleSortTokensPerThread; ++i) {
        const bool mine = (own_bits >> i) & 1;
        // the inverse of the list, for the reduce that adds up the rows coming back: where is (token, rank)?
        if (row_of_pair != nullptr && i < tokens_per_thread && first + i < num_tokens)
            row_of_pair[int64_t(first + i) * num_ranks + r] = mine ? int32_t(pos) : -1;
        if (mine) sorted_token_ids[pos++] = first + i;
    }
    if (tid == 0) {
        send_counts[r] = total;
        send_cumsum[r] = base;
        if (r == num_ranks - 1) send_cumsum[num_ranks] = int64_t(base) + total;
    }
    report_done(report, int64_t(base) + total);  // the last rank's end is the total
}

// ---------------------------------------------------------------------
// The same sort in one launch for a multiple of 8 ranks up to 64 and a matrix of up to 512 KB.  One workgroup per 256
// tokens; each reads the whole matrix (from L2), 8 ranks of a token per 8-byte word, adding the bool bytes of a
// word up eight at a time, once over all tokens and once over those before its own: the first gives where every
// rank's ids begin, the second where its own tokens' ids do.  Against one workgroup per rank, a token's row of
// row_of_pair is written in one piece, and the loads are independent of one another; against three launches
// (count, scan, scatter) it is one.  What bounds it are the instructions of sixteen waves on one compute unit, so what a
// wave need not do by itself is shared: the lanes' counts of all waves are added up in LDS, and each wave sums a few of the
// columns over the lanes (every wave for itself, two ranks at a time, took 12.2 us for 4096 tokens to 32 ranks); bytes are
// taken for the 0 and 1 of a bool, which one test at the end confirms; only the waves that are asked count the own tokens.
// ---------------------------------------------------------------------
constexpr int kWideSortTokens = 256;  // tokens per workgroup
constexpr int kWideSortThreads = 1024;
constexpr int64_t kWideSortMaxBytes = 512 * 1024;

// A token's row of kWords words out of the matrix as a buffer: zeros past its end.
template <int kWords>
__device__ __forceinline__ void load_member_words(__amdgpu_buffer_rsrc_t matrix, int t, uint64_t (&row)[kWords]) {
    const int at = t * (kWords * 8);
#pragma unroll
    for (int q = 0; q + 1 < kWords; q += 2) {
        const u32x4 v = load_row_u32x4<false>(matrix, at + q * 8);
        row[q] = (uint64_t(v[1]) << 32) | v[0], row[q + 1] = (uint64_t(v[3]) << 32) | v[2];
    }
    if constexpr (kWords % 2 != 0) {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(matrix, at + (kWords - 1) * 8, 0, 0);
        row[kWords - 1] = (uint64_t(v[1]) << 32) | v[0];
    }
}

// all[q] (bytes) += the members among this thread's tokens tid, tid + 1024, ..., before[q] those among them in front of
// token `begin`, a multiple of 256.  kBool: bytes are 0 or 1; returns whether they were.
template <int kWords, bool kBool>
__device__ __forceinline__ bool count_members(__amdgpu_buffer_rsrc_t matrix, int num_tokens, int begin,
                                              uint64_t (&all)[kWords], uint64_t (&before)[kWords]) {
    constexpr int kAhead = kWords <= 4 ? 4 : 2;  // tokens in flight
    const int tid = threadIdx.x;
    uint64_t bits = 0;
#pragma unroll
    for (int q = 0; q < kWords; ++q) all[q] = before[q] = 0;
    for (int t0 = 0; t0 < num_tokens; t0 += kAhead * kWideSortThreads) {
        uint64_t v[kAhead][kWords];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load_member_words(matrix, t0 + u * kWideSortThreads + tid, v[u]);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int round = t0 + u * kWideSortThreads;
            if constexpr (!kBool)
#pragma unroll
                for (int q = 0; q < kWords; ++q) v[u][q] = nonzero_bytes(v[u][q]);
            if (round == begin / kWideSortThreads * kWideSortThreads)  // once: what came before it is all there
#pragma unroll
                for (int q = 0; q < kWords; ++q) before[q] = all[q] + (round + tid < begin ? v[u][q] : 0);
#pragma unroll
            for (int q = 0; q < kWords; ++q) {
                all[q] += v[u][q];
                if constexpr (kBool) bits |= v[u][q];
            }
        }
    }
    return __ballot((bits & 0xfefefefefefefefeull) != 0) == 0;
}

template <int kWords>  // 8-byte words of a token's row: ranks / 8
__global__ __launch_bounds__(kWideSortThreads) void routing_sort_wide_kernel(
    const uint8_t* __restrict__ is_token_in_rank, int num_tokens, int32_t* __restrict__ send_counts,
    int64_t* __restrict__ send_cumsum, int64_t* __restrict__ sorted_token_ids, int32_t* __restrict__ row_of_pair,
    int64_t* __restrict__ report) {
    constexpr int kThreads = kWideSortThreads;
    constexpr int kRanks = kWords * 8, kWaves = kThreads / kWave;
    constexpr int kTokenWaves = kWideSortTokens / kWave, kRankShares = kWaves / kTokenWaves;
    constexpr int kColumns = kWords * 2;  // even and odd bytes of a word, widened to 16 bits
    __shared__ unsigned long long lane_counts[2][kColumns][kWave];  // over all tokens, and over those before
    __shared__ int32_t rank_counts[2][kRanks];
    __shared__ int32_t start[kRanks];                // where the ids of this workgroup's tokens begin, per rank
    __shared__ int32_t chunk_cnt[kTokenWaves][kRanks];
    __shared__ int32_t total_of_all;
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block();
    const int begin = blockIdx.x * kWideSortTokens;
    const auto matrix = row_buffer(is_token_in_rank, num_tokens * kRanks);
    // this thread's own token, loaded with the rest: wave w has tokens (w % 4) * 64 + lane
    const int tw = w & (kTokenWaves - 1), share = w / kTokenWaves;
    const int own = begin + tw * kWave + lane;
    uint64_t own_row[kWords];
    load_member_words(matrix, own, own_row);
    for (int i = tid; i < 2 * kColumns * kWave; i += kThreads) (&lane_counts[0][0][0])[i] = 0;
    lds_barrier();
    uint64_t all[kWords], before[kWords];
    if (!count_members<kWords, true>(matrix, num_tokens, begin, all, before))
        count_members<kWords, false>(matrix, num_tokens, begin, all, before);
#pragma unroll
    for (int q = 0; q < kWords; ++q)
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) {
            atomicAdd(&lane_counts[0][q * 2 + odd][lane], (all[q] >> (8 * odd)) & 0x00ff00ff00ff00ffull);
            if (begin > 0) atomicAdd(&lane_counts[1][q * 2 + odd][lane], (before[q] >> (8 * odd)) & 0x00ff00ff00ff00ffull);
        }
    if (share == 0) {  // this workgroup's own tokens per rank and wave
        int mine = 0;
#pragma unroll
        for (int q = 0; q < kWords; ++q)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int votes = __popcll(__ballot(((own_row[q] >> (8 * i)) & 0xff) != 0));
                if (lane == q * 8 + i) mine = votes;
            }
        if (lane < kRanks) chunk_cnt[tw][lane] = mine;
    }
    lds_barrier();
#pragma unroll
    for (int c = w; c < 2 * kColumns; c += kWaves) {
        const int which = c / kColumns, column = c % kColumns;
        const uint64_t counts = lane_counts[which][column][lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int sum = wave_inclusive_sum(int((counts >> (16 * i)) & 0xffff));
            if (lane == kWave - 1) rank_counts[which][column / 2 * 8 + 2 * i + column % 2] = sum;
        }
    }
    lds_barrier();
    if (w == 0) {
        const int total = lane < kRanks ? rank_counts[0][lane] : 0;
        const int incl = wave_inclusive_sum(total);
        if (lane < kRanks) start[lane] = incl - total + rank_counts[1][lane];
        if (lane == kRanks - 1) total_of_all = incl;
        if (blockIdx.x == 0) {
            if (lane == kRanks - 1) send_cumsum[kRanks] = incl;
            if (lane < kRanks) send_counts[lane] = total, send_cumsum[lane] = incl - total;
        }
    }
    lds_barrier();
    // wave (share, tw) writes its 64 tokens' places in its share of the ranks
    constexpr int kPerShare = kRanks / kRankShares;
    int place[kPerShare];
#pragma unroll
    for (int i = 0; i < kPerShare; ++i) {
        const int r = share * kPerShare + i;
        uint64_t word = 0;  // own_row[r / 8] with an index the compiler can resolve
#pragma unroll
        for (int q = 0; q < kWords; ++q)
            if (q == (r >> 3)) word = own_row[q];
        const bool in = ((word >> (8 * (r & 7))) & 0xff) != 0;
        const uint64_t votes = __ballot(in);
        int pos = start[r] + __popcll(votes & lanes_below(lane));
#pragma unroll
        for (int t2 = 0; t2 < kTokenWaves - 1; ++t2) pos += t2 < tw ? chunk_cnt[t2][r] : 0;
        if (in) sorted_token_ids[pos] = own;
        place[i] = in ? pos : -1;
    }
    if (row_of_pair != nullptr) {
        const auto places = row_buffer(reinterpret_cast<const uint8_t*>(row_of_pair), num_tokens * (kRanks * 4));
        const int at = own * (kRanks * 4) + share * (kPerShare * 4);
#pragma unroll
        for (int i = 0; i + 3 < kPerShare; i += 4)
            store_row_u32x4<false>(places, at + i * 4,
                                   u32x4{uint32_t(place[i]), uint32_t(place[i + 1]), uint32_t(place[i + 2]), uint32_t(place[i + 3])});
        if constexpr (kPerShare % 4 != 0)  // two
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{uint32_t(place[kPerShare - 2]), uint32_t(place[kPerShare - 1])}, places,
                                                  at + (kPerShare - 2) * 4, 0, 0);
    }
    report_done(report, total_of_all);
}

// ---------------------------------------------------------------------
// channel_prefix_matrix: one workgroup per destination rank, one wave per
// channel (up to sixteen at a time), then an in-place prefix over channels.
// Reference: csrc/kernels/intranode.cu:90-112.
// ---------------------------------------------------------------------
__global__ __launch_bounds__(1024) void channel_prefix_kernel(const uint8_t* __restrict__ is_token_in_rank,
                                                              int num_tokens, int num_ranks, int num_channels,
                                                              int32_t* __restrict__ cpm) {
    extern __shared__ int32_t per_channel[];  // [C]
    const int dst = blockIdx.x, lane = lane_id(), w = wave_in_block();
    const int waves = block_threads() >> 6;
    const int per = (num_tokens + num_channels - 1) / num_channels;
    for (int ch = w; ch < num_channels; ch += waves) {
        const int begin = min(per * ch, num_tokens), end = min(begin + per, num_tokens);
        int count = 0;
        for (int t0 = begin + lane; t0 < end; t0 += kWave * 8) {  // eight loads in flight per lane
            uint8_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = t0 + u * kWave;
                v[u] = t < end ? is_token_in_rank[int64_t(t) * num_ranks + dst] : uint8_t(0);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) count += v[u] != 0;
        }
        count = wave_sum(count);
        if (lane == 0) per_channel[ch] = count;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int ch = 0; ch < num_channels; ++ch) {
            run += per_channel[ch];
            cpm[int64_t(dst) * num_channels + ch] = run;
        }
    }
}

// The same for a multiple of 8 ranks: one workgroup per 8 of them, so a wave reads the membership of eight ranks
// with one 8-byte load per token, up to sixteen of them in flight, and adds the bool bytes up eight at a time.  The
// bytes of a row that eight workgroups used to fetch for themselves are fetched once; the sums of eight ranks are
// eight times the work of one's.
// Instructions bound it where channels are long: the bytes are taken for the 0 and 1 of a bool, which one test a channel
// confirms (4096 tokens 3.8 -> 3.4 us, 12000 5.6 -> 4.5).
template <int kAhead, bool kBool>
__device__ __forceinline__ bool count_channel(const uint64_t* __restrict__ is_token_in_rank, int begin, int end, int q,
                                              int num_words, int (&count)[8]) {
    const int lane = lane_id();
    uint64_t bits = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) count[i] = 0;
    for (int t0 = begin + lane; t0 - lane < end; t0 += kWave * kAhead) {
        uint64_t v[kAhead], sum = 0;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int t = t0 + u * kWave;
            v[u] = is_token_in_rank[int64_t(t < end ? t : end - 1) * num_words + q];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const uint64_t one = t0 + u * kWave < end ? (kBool ? v[u] : nonzero_bytes(v[u])) : 0;
            sum += one;
            if constexpr (kBool) bits |= one;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)  // bytes widened to 16 bits: 64 lanes of at most 16 fit
#pragma unroll
            for (int odd = 0; odd < 2; ++odd) {
                const int part = int((uint32_t(sum >> (32 * half)) >> (8 * odd)) & 0x00ff00ffu);
                const uint32_t all = uint32_t(__builtin_amdgcn_readlane(wave_inclusive_sum(part), kWave - 1));
                count[half * 4 + odd] += int(all & 0xffffu);
                count[half * 4 + odd + 2] += int(all >> 16);
            }
    }
    return __ballot((bits & 0xfefefefefefefefeull) != 0) == 0;
}

template <int kAhead>  // loads in flight per lane: 4 for channels of up to 256 tokens, else 16
__global__ __launch_bounds__(1024) void channel_prefix_words_kernel(const uint64_t* __restrict__ is_token_in_rank,
                                                                    int num_tokens, int num_words, int num_channels,
                                                                    int32_t* __restrict__ cpm) {
    extern __shared__ int32_t per_channel[];  // [C][8]
    const int q = blockIdx.x, lane = lane_id(), w = wave_in_block();
    const int waves = block_threads() >> 6;
    const int per = (num_tokens + num_channels - 1) / num_channels;
    for (int ch = w; ch < num_channels; ch += waves) {
        const int begin = min(per * ch, num_tokens), end = min(begin + per, num_tokens);
        int count[8];
        if (!count_channel<kAhead, true>(is_token_in_rank, begin, end, q, num_words, count))
            count_channel<kAhead, false>(is_token_in_rank, begin, end, q, num_words, count);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (lane == i) per_channel[ch * 8 + i] = count[i];
    }
    lds_barrier();
    if (threadIdx.x < 8) {
        int run = 0;
        for (int ch = 0; ch < num_channels; ++ch) {
            run += per_channel[ch * 8 + threadIdx.x];
            cpm[int64_t(q * 8 + threadIdx.x) * num_channels + ch] = run;
        }
    }
}

// ---------------------------------------------------------------------
// pack_rows: dst[i] = src[ids[i]].  One workgroup per output row, two 16-byte
// vectors per thread in flight (wider rows loop).  The row
// count is read from device memory so no host sync is needed.
// Reference: deep_ep/buffer.py:877,917 (torch advanced-index gathers).
//
// It is bound by HBM, and by which bytes get there.  A row goes to several
// ranks, and in list order (rank by rank) its copies are a whole pass over the
// source apart: every pass reads the source again.  kGrouped takes the list as
// the merge of its ranks' lists instead: group g is the g-th of 2^group_log2
// equal parts of every rank's list, which are about the same tokens because
// each list ascends, and workgroups 8 apart -- on one XCD, sharing an L2 -- work
// through one group, so a source row is read once and found in that L2 by the
// other ranks.  Any routing gives the same result; a skewed one only shares less.
// Past 48 MB the packed rows are stored with the non-temporal hint: otherwise they push the source rows, and
// whatever the caches hold of others, out again.  What reads them next is a transport, at the rate of its links, to which
// the memory-side cache (256 MB) is worth nothing; a copy on this GPU would find them there and take back what the hint
// gives.  Microseconds of pack and pack + copy of the packed rows, ordinary stores against the hint (R = 8, four sets of
// tensors in turn):
//    19 MB   7.0 / 5.0    13.8 / 15.3     118 MB  35.7 / 21.7   72.4 / 78.0
//    39 MB  10.0 / 8.9    25.6 / 29.5     129 MB  40.4 / 23.2   83.8 / 85.6
//    78 MB  24.0 / 15.3   48.8 / 54.2     140 MB  42.0 / 25.3   93.9 / 91.4
//    97 MB  29.3 / 18.4   59.8 / 65.7     155 MB  48.5 / 27.4  107.2 / 102.5    311 MB  88.7 / 54.6  209 / 197
// Grouping and hint against list order and ordinary stores: 12289 x 14336 bytes (934 MB) 305 -> 211 us, 4096 x 7168
// (155 MB) 48.1 -> 27.3.  Rows as buffers, and the scales fetched with the payload instead of behind its stores (a wave
// of their own takes the place of payload: 28.6 -> 30.5 us for 4096 x 7168): 202 -> 188 us (5.9 TB/s on the bytes that
// have to move), 9000 x 10240 to 32 ranks 151 -> 136, 4096 x 7168 27.4 -> 27.1.  Four trips to memory stand in front of a
// row here, which takes more rows in flight to hide than the copies of described rows need: two vectors a thread
// against one, 205 and 273 us for 512 threads and for whole rows; three or four 186 to 195, and 28.4 and 29.5 for rows
// of 7168 bytes.
// Groups of 6, 12, 24 and 48 MB: 230, 215, 211 and 207 us, but much is lost where their source rows no longer fit an L2
// (4 MB; of a source larger than what is packed, no more than that is read: 896 rows out of 3.1 GB 7.5 -> 5.9 us, 20000
// 86 -> 83): a whole prefill of 9000 x 7168 in fp8 to 8 ranks 262 us with 4.0 MB of source a group and 250 with 2.0, of 6000 x
// 14336 at top-6 188 and 173 with 5.4 and 2.7, of 7000 x 8192 127.3 and 125 with 3.4 and 1.7; 2.9 at 32 ranks gains (308
// -> 302 against half).  Fewer than two groups an XCD lose a tenth, and two of more than 16 MB some: the pack of 7000 x 7168
// in fp8 to 32 ranks behind its cast 68.5 us with 16 groups of 22 MB, 63.6 with 32.  Against 8 to 128 groups by force, 1500
// to 12000 rows of 2 to 14 KB, 3.3 to 7.3 copies: past 128 MB these bounds are within 2 % of the best everywhere; below,
// on four sets of tensors in turn, 8 groups are up to 96 MB (7168 x 8 ranks: 72 MB 17.4 us and 18.6 with 16, 88 MB 21.7 and
// 22.6) and lose beyond (112 MB 30.5 and 28.0).  The groups' rows drift apart by some fifty
// tokens, so a group reads half as much again as its share of the source.
// Up to 256 threads up to 50 MB of packed rows, then 512.  Rows of 14336 bytes to 8 ranks, four sets of tensors in turn, 512
// / 256 threads, and the same with a copy of the packed rows behind it: 36 MB 9.0 / 8.7 us, 21.7 / 22.8; 45 MB 10.6 / 10.2,
// 26.3 / 27.5; 54 MB 11.6 / 12.9; 60 MB 13.7 / 15.5, 33.4 / 34.7; 80 MB 18.8 / 19.7, 43.7 / 44.3; 95 MB 23.7 / 24.2, 54.8 / 53.0;
// 111 MB 27.1 / 28.2, 65.0 / 63.3; rows of 8704 to 28672 bytes alike (51 MB of 8704 11.3 / 10.2, 54 MB 12.6 / 12.7), narrower ones have
// 256 either way.  A whole prefill on three sets of buffers in turn, hint past 128 MB / past 48: 1000 x 14336 bytes (72 MB)
// 63.0 / 59.1 us, 2000 x 7168 (73 MB) 90.2 / 83.6 (with the reduce's), 4000 x 4096 to 16 ranks (98 MB) 80.8 / 77.9; past 24: the
// same.  In list order, where the rows stream, the
// same threads move one vector at a time: two trips to memory stand in front of a row there.  4096 x 14336 88.5 us against 96.1
// with two vectors in flight, 4096 x 7168 45.5 and 47.9 (46.0 to 48 with twice the threads), 12289 x 14336 258 and 267; against
// two vectors and ordinary stores 60 MB 17.3 and 18.4, 80 MB 22.6 and 24.0, 110 MB 31.0 and 34.4.
// ---------------------------------------------------------------------
constexpr int64_t kPackGroupBytes = int64_t(12) << 20;  // packed bytes of one of 8 groups; 16 MB of 16, 24 MB of more
constexpr int64_t kPackSourceBytes = int64_t(3) << 20;  // source bytes of a group
constexpr int64_t kPackStreamBytes = int64_t(48) << 20;
constexpr int64_t kPackSmallBytes = int64_t(50) << 20;

struct PackArgs {
    const uint8_t* src;
    uint8_t* dst;
    int num_src_rows, row_bytes, threads;
    const uint8_t* scale_src;
    uint8_t* scale_dst;
    int scale_row_bytes;
};

template <bool kStream, int kVecs>
__device__ __forceinline__ void pack_row(const PackArgs& a, const int64_t* __restrict__ ids, int64_t row) {
    const int64_t id = ids[row];
    if (id < 0 || id >= a.num_src_rows) return;
    const int tid = threadIdx.x;
    const uint32_t* scales = reinterpret_cast<const uint32_t*>(a.scale_src + id * a.scale_row_bytes);
    uint32_t* scales_to = reinterpret_cast<uint32_t*>(a.scale_dst + row * a.scale_row_bytes);
    const int num_scales = a.scale_src != nullptr ? a.scale_row_bytes / 4 : 0;
    uint32_t scale = 0;
    if (tid < num_scales) scale = scales[tid];  // in flight with the payload, not behind its stores
    block_copy_row<kVecs, false, kStream>(a.src + id * a.row_bytes, a.dst + row * a.row_bytes, a.row_bytes / 16, tid, a.threads);
    if (tid < num_scales) scales_to[tid] = scale;
    for (int v = tid + a.threads; v < num_scales; v += a.threads) scales_to[v] = scales[v];
}

template <bool kStream>
__global__ __launch_bounds__(1024) void pack_rows_kernel(const int64_t* __restrict__ num_rows_dev,
                                                         const int64_t* __restrict__ ids, int64_t max_rows,
                                                         uint32_t grid, PackArgs a) {
    int64_t num_rows = *num_rows_dev;
    if (num_rows > max_rows) num_rows = max_rows;
    for (int64_t i = blockIdx.x; i < num_rows; i += grid) pack_row<kStream, kStream ? 1 : 2>(a, ids, i);
}

template <bool kStream>
__global__ __launch_bounds__(1024) void pack_groups_kernel(const int64_t* __restrict__ cumsum,
                                                           const int64_t* __restrict__ ids, int64_t max_rows,
                                                           int num_ranks, int group_log2, uint32_t slots, PackArgs a) {
    const int lane = lane_id();
    const uint32_t xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
    const uint32_t g = i / slots * 8 + xcd;
    // lane r: the part of rank r's list that is in the group
    int64_t first = 0;
    int skip = 0, size = 0;
    if (lane < num_ranks) {
        first = lane == 0 ? 0 : cumsum[lane];  // the list starts at its first row, whatever cumsum[0] is
        const int64_t n = cumsum[lane + 1] - first;
        skip = int((n * g) >> group_log2);
        size = int((n * (g + 1)) >> group_log2) - skip;
    }
    const int incl = wave_inclusive_sum(size);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    const int64_t begin = first + skip - (incl - size);  // list row of slot s of the group: begin + s
    for (int slot = i % slots; slot < total; slot += slots) {
        const int r = __popcll(__ballot(incl <= slot));  // lanes past the ranks hold the total
        const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(begin), r);
        const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(begin >> 32), r);
        const int64_t row = int64_t((uint64_t(hi) << 32) | lo) + slot;
        if (row >= 0 && row < max_rows) pack_row<kStream, 2>(a, ids, row);
    }
}

}  // namespace deepep

using namespace deepep;

extern "C" {

size_t deepep_layout_workspace_bytes(int num_tokens, int num_ranks, int num_experts) {
    const int64_t blocks = (int64_t(num_tokens) + kLayoutThreads - 1) / kLayoutThreads;
    const int64_t width = int64_t(num_experts) + num_ranks + num_ranks / 8 + 1;
    return size_t((blocks < 1 ? 1 : blocks) * width * 4);
}

int deepep_get_dispatch_layout(const int64_t* topk_idx, int num_tokens, int num_topk, int num_ranks,
                               int num_experts, int32_t* num_tokens_per_rank, int32_t* num_tokens_per_rdma_rank,
                               int32_t* num_tokens_per_expert, uint8_t* is_token_in_rank, void* workspace,
                               size_t workspace_bytes, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_tokens >= 0 && num_topk > 0);
    EP_HOST_ASSERT(num_experts > 0);
    EP_HOST_ASSERT(num_ranks > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(num_ranks <= 64 * kMaxRankWords);
    EP_HOST_ASSERT(num_tokens_per_rdma_rank == nullptr || (num_ranks % 8 == 0 && num_ranks > 8));
    EP_HOST_ASSERT(num_tokens_per_rank != nullptr && num_tokens_per_expert != nullptr);
    EP_HOST_ASSERT(num_tokens == 0 || (topk_idx != nullptr && is_token_in_rank != nullptr));
    EP_HOST_ASSERT((num_ranks & 7) != 0 || (reinterpret_cast<uintptr_t>(is_token_in_rank) & 7) == 0);
    const int num_nodes = num_tokens_per_rdma_rank != nullptr ? num_ranks / 8 : 0;
    const int width = num_experts + num_ranks + num_nodes;
    EP_HOST_ASSERT(size_t(width) * 4 <= 64 * 1024);
    const int partials = num_tokens == 0 ? 1 : (num_tokens + kLayoutThreads - 1) / kLayoutThreads;
    EP_HOST_ASSERT(workspace != nullptr && workspace_bytes >= size_t(partials) * width * 4);
    const int blocks = num_tokens <= layout_one_block_tokens(num_ranks, num_topk) ? 1 : partials;
    const int threads = blocks == 1 && num_tokens > kLayoutThreads ? kLayoutOneBlockThreads : kLayoutThreads;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    int32_t* partial = reinterpret_cast<int32_t*>(workspace);
    const uint32_t experts_per_rank = uint32_t(num_experts / num_ranks);
    EP_HOST_ASSERT(num_experts < 65536);
    const uint32_t rank_magic =
        experts_per_rank == 1 ? 0u : uint32_t(((uint64_t(1) << 32) + experts_per_rank - 1) / experts_per_rank);
#define DEEPEP_LAUNCH_LAYOUT(WORDS)                                                                              \
    launch(layout_count_kernel<WORDS>, blocks, threads, size_t(width) * 4, s,                                         \
        topk_idx, num_tokens, num_topk, num_ranks, num_experts, rank_magic, num_nodes, is_token_in_rank, partial, \
        num_tokens_per_rank, num_tokens_per_rdma_rank, num_tokens_per_expert)
    if (num_ranks <= kWave) DEEPEP_LAUNCH_LAYOUT(1);
    else DEEPEP_LAUNCH_LAYOUT(kMaxRankWords);
#undef DEEPEP_LAUNCH_LAYOUT
    EP_LAUNCH_CHECK();
    if (blocks == 1) return 0;
    launch(layout_reduce_kernel, (width + kLayoutThreads - 1) / kLayoutThreads, kLayoutThreads, 0, s,
        partial, blocks, num_experts, num_ranks, num_nodes, num_tokens_per_rank, num_tokens_per_rdma_rank,
        num_tokens_per_expert);
    EP_LAUNCH_CHECK();
    return 0;
}

size_t deepep_routing_sort_workspace_bytes(int num_tokens, int num_ranks) {
    const int64_t chunks = (int64_t(num_tokens) + kSortChunk - 1) / kSortChunk;
    return size_t((chunks < 1 ? 1 : chunks) * num_ranks * 4);
}

// Which form sorts.  Microseconds of the wide form against one workgroup per rank, with row_of_pair:
//   ranks       8            16           24           32            48            64
//   512 tokens  3.3 / 2.9    4.0 / 3.2    5.4 / 3.5    5.8 /  3.7     7.8 /  4.2     9.6 /  5.5
//   1024        3.3 / 3.4    4.0 / 3.6    5.4 / 3.8    5.8 /  4.0     7.8 /  4.6     9.7 /  5.6
//   1536        3.3 / 3.8    4.0 / 4.2    5.4 / 4.6    5.9 /  5.1     7.9 /  7.1    10.0 / 10.0
//   2047        3.3 / 4.2    4.1 / 4.7    5.4 / 5.2    5.9 /  5.9     8.0 /  8.5    10.1 / 12.7
//   3000        3.3 / 4.4    4.1 / 5.9    5.5 / 6.9    5.9 /  8.7     8.4 / 13.1    11.4 / 17.1
//   8192        3.9 / 10.0   4.7 / 15.0   6.7 / 20     7.0 / 23.2                   15.8 / 41.7
// Upwards every workgroup reads the whole matrix: at 512 KB that still beats the three launches (8 ranks, 20000 tokens
// 7.2 against 16.5 before the wide form's own time was halved; 24 ranks, 12289 7.8 against 34.2), past that its work
// grows with the square of the batch.
static bool sort_is_wide(const uint8_t* is_token_in_rank, int num_tokens, int num_ranks) {
    // (up to 2048 tokens a thread of one workgroup per rank has two: 24 ranks 5.7 / 5.5, 40 ranks 7.8 / 7.4, 56 ranks 10.1 / 10.6)
    const int from = num_ranks == 8 ? 1024 : num_ranks == 16 ? 1280 : num_ranks == 24 || num_ranks == 40 ? 2049 : 2048;
    return num_ranks % 8 == 0 && num_ranks <= 64 && (reinterpret_cast<uintptr_t>(is_token_in_rank) & 7) == 0 &&
           num_tokens >= from && int64_t(num_tokens) * num_ranks <= kWideSortMaxBytes;
}
static bool sort_is_single(int num_tokens, int num_ranks) {
    return num_tokens <= kSortChunk * kSingleSortTokensPerThread && num_ranks <= 64;
}

int deepep_routing_sort_report_words(const uint8_t* is_token_in_rank, int num_tokens, int num_ranks) {
    if (sort_is_wide(is_token_in_rank, num_tokens, num_ranks)) return (num_tokens + kWideSortTokens - 1) / kWideSortTokens;
    if (sort_is_single(num_tokens, num_ranks)) return num_ranks;
    return num_tokens <= 0 ? 1 : (num_tokens + kSortChunk - 1) / kSortChunk;
}

int deepep_moe_routing_sort_reporting(const uint8_t* is_token_in_rank, int num_tokens, int num_ranks,
                                      int64_t* sorted_token_ids, int32_t* send_counts, int64_t* send_cumsum,
                                      int32_t* row_of_pair, int64_t* report_host, void* workspace,
                                      size_t workspace_bytes, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_tokens >= 0 && num_ranks > 0 && num_ranks <= 1024);
    EP_HOST_ASSERT(send_counts != nullptr && send_cumsum != nullptr);
    EP_HOST_ASSERT(num_tokens == 0 || (is_token_in_rank != nullptr && sorted_token_ids != nullptr));
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(report_host) & 7) == 0);
    const int chunks = num_tokens == 0 ? 1 : (num_tokens + kSortChunk - 1) / kSortChunk;
    EP_HOST_ASSERT(workspace != nullptr && workspace_bytes >= size_t(chunks) * num_ranks * 4);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (sort_is_wide(is_token_in_rank, num_tokens, num_ranks)) {
        const int blocks = (num_tokens + kWideSortTokens - 1) / kWideSortTokens;
#define DEEPEP_LAUNCH_SORT(WORDS)                                                                  \
    case WORDS:                                                                                    \
        launch(routing_sort_wide_kernel<WORDS>, blocks, kWideSortThreads, 0, s,                        \
            is_token_in_rank, num_tokens, send_counts, send_cumsum, sorted_token_ids, row_of_pair, report_host); \
        break
        switch (num_ranks / 8) {
            DEEPEP_LAUNCH_SORT(1);
            DEEPEP_LAUNCH_SORT(2);
            DEEPEP_LAUNCH_SORT(3);
            DEEPEP_LAUNCH_SORT(4);
            DEEPEP_LAUNCH_SORT(5);
            DEEPEP_LAUNCH_SORT(6);
            DEEPEP_LAUNCH_SORT(7);
            DEEPEP_LAUNCH_SORT(8);
        }
#undef DEEPEP_LAUNCH_SORT
        EP_LAUNCH_CHECK();
        return 0;
    }
    if (sort_is_single(num_tokens, num_ranks)) {
#define DEEPEP_LAUNCH_SORT(THREADS)                                                                            \
    launch(routing_sort_single_kernel<THREADS>, num_ranks, THREADS, 0, s,                                           \
        is_token_in_rank, num_tokens, num_ranks, num_tokens == 0 ? 1 : (num_tokens + THREADS - 1) / THREADS,    \
        send_counts, send_cumsum, sorted_token_ids, row_of_pair, report_host)
        if (num_tokens <= kSmallSortTokens) DEEPEP_LAUNCH_SORT(256);
        else DEEPEP_LAUNCH_SORT(kSortChunk);
#undef DEEPEP_LAUNCH_SORT
        EP_LAUNCH_CHECK();
        return 0;
    }
    int32_t* table = reinterpret_cast<int32_t*>(workspace);
    const size_t lds = size_t(kSortChunk / kWave) * num_ranks * 4;
    launch(routing_sort_pass_kernel<false>, chunks, kSortChunk, lds, s, is_token_in_rank, num_tokens, num_ranks, table,
                                                                    sorted_token_ids, nullptr, nullptr, nullptr);
    EP_LAUNCH_CHECK();
    launch(routing_sort_scan_kernel, 1, 256, size_t(num_ranks + 1) * 8, s, table, chunks, num_ranks, send_counts,
                                                                       send_cumsum,
                                                                       num_tokens == 0 ? report_host : nullptr);
    EP_LAUNCH_CHECK();
    if (num_tokens > 0) {
        launch(routing_sort_pass_kernel<true>, chunks, kSortChunk, lds, s, is_token_in_rank, num_tokens, num_ranks,
                                                                       table, sorted_token_ids, row_of_pair,
                                                                       send_cumsum + num_ranks, report_host);
        EP_LAUNCH_CHECK();
    }
    return 0;
}

int deepep_moe_routing_sort(const uint8_t* is_token_in_rank, int num_tokens, int num_ranks,
                            int64_t* sorted_token_ids, int32_t* send_counts, int64_t* send_cumsum,
                            int32_t* row_of_pair, void* workspace, size_t workspace_bytes, void* stream) {
    return deepep_moe_routing_sort_reporting(is_token_in_rank, num_tokens, num_ranks, sorted_token_ids, send_counts,
                                             send_cumsum, row_of_pair, nullptr, workspace, workspace_bytes, stream);
}

int deepep_channel_prefix_matrix(const uint8_t* is_token_in_rank, int num_tokens, int num_ranks, int num_channels,
                                 int32_t* channel_prefix_matrix, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_tokens >= 0 && num_ranks > 0 && num_channels > 0 && num_channels <= 4096);
    EP_HOST_ASSERT(channel_prefix_matrix != nullptr);
    EP_HOST_ASSERT(num_tokens == 0 || is_token_in_rank != nullptr);
    // one wave per channel, up to sixteen at a time
    const int threads = num_channels >= 16 ? 1024 : ((num_channels + 3) / 4) * 256;
    // Eight ranks a workgroup pays once there is enough to fetch, and not for so many ranks that their workgroups fill
    // the chip anyway.  Microseconds behind the launch that writes the matrix, against one rank a workgroup:
    //   ranks                       8           16          32          64
    //   131 tokens, 10 channels     2.4 / 2.4   2.7 / 2.4   2.8 / 2.6   3.0 / 2.7
    //   1024, 24 channels           3.1 / 3.1   3.8 / 3.3   3.7 / 3.3   4.1 / 3.4
    //   2048, 16 channels           2.7 / 2.7   2.8 / 2.8   3.1 / 3.3   4.1 / 4.0
    //   4096, 24 channels           3.5 / 4.1   3.8 / 4.3   3.9 / 4.9   5.0 / 5.3
    //   12289, 10 channels          5.7 / 7.9   6.0 / 8.0   7.7 / 8.9  11.2 / 10.1
    const bool by_words = num_ranks == 8 || (num_ranks % 8 == 0 && num_ranks <= 32 && num_tokens >= 2048);
    if (by_words && (reinterpret_cast<uintptr_t>(is_token_in_rank) & 7) == 0 && num_channels <= 1024) {
#define DEEPEP_LAUNCH_CHANNELS(AHEAD)                                                                              \
    launch(channel_prefix_words_kernel<AHEAD>, num_ranks / 8, threads, size_t(num_channels) * 32,                        \
                                         reinterpret_cast<hipStream_t>(stream),                                  \
        reinterpret_cast<const uint64_t*>(is_token_in_rank), num_tokens, num_ranks / 8, num_channels,              \
        channel_prefix_matrix)
        if ((int64_t(num_tokens) + num_channels - 1) / num_channels <= 4 * kWave) DEEPEP_LAUNCH_CHANNELS(4);
        else DEEPEP_LAUNCH_CHANNELS(16);
#undef DEEPEP_LAUNCH_CHANNELS
        EP_LAUNCH_CHECK();
        return 0;
    }
    launch(channel_prefix_kernel, num_ranks, threads, size_t(num_channels) * 4, reinterpret_cast<hipStream_t>(stream),
        is_token_in_rank, num_tokens, num_ranks, num_channels, channel_prefix_matrix);
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_pack_rows_by_rank(const void* src, const void* scale_src, const int64_t* sorted_token_ids,
                             const int64_t* num_rows_dev, const int64_t* send_cumsum, int num_ranks, int64_t max_rows,
                             int num_src_rows, int row_bytes, int scale_row_bytes, void* dst, void* scale_dst,
                             void* stream) {
    clear_error();
    EP_HOST_ASSERT(max_rows >= 0 && num_src_rows >= 0);
    EP_HOST_ASSERT(row_bytes > 0 && row_bytes % 16 == 0);
    EP_HOST_ASSERT(scale_src == nullptr || (scale_dst != nullptr && scale_row_bytes > 0 && scale_row_bytes % 4 == 0));
    EP_HOST_ASSERT(send_cumsum == nullptr || num_ranks > 0);
    if (max_rows == 0) return 0;
    EP_HOST_ASSERT(src != nullptr && dst != nullptr && sorted_token_ids != nullptr && num_rows_dev != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(src) & 15) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(scale_src) & 3) == 0 && (reinterpret_cast<uintptr_t>(scale_dst) & 3) == 0);
    PackArgs a;
    a.src = reinterpret_cast<const uint8_t*>(src), a.scale_src = reinterpret_cast<const uint8_t*>(scale_src);
    a.num_src_rows = num_src_rows, a.row_bytes = row_bytes, a.scale_row_bytes = scale_row_bytes;
    a.dst = reinterpret_cast<uint8_t*>(dst), a.scale_dst = reinterpret_cast<uint8_t*>(scale_dst);
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    const bool stream_rows = max_rows * row_bytes > kPackStreamBytes;
    // Below a group's worth of packed rows everything stays in the caches and the grouping's lookup is one more
    // round trip in front of the rows: 6.5 MB 2.9 us against 3.4, 12 MB 3.9 either way, 22 MB 6.7 against 5.0.
    // A wave holds the ranks' parts one a lane, hence the 64.
    const bool grouped =
        send_cumsum != nullptr && num_ranks > 1 && num_ranks <= kWave && max_rows * row_bytes > kPackGroupBytes;
    a.threads = flat_row_threads((row_bytes / 16 + 1) / 2, max_rows * row_bytes > kPackSmallBytes ? 512 : 256);
    const int threads = a.threads;
    if (grouped) {
        int group_log2 = 3;  // the fewer groups an XCD, the smaller, and no group's source rows larger than fit its L2
        const int64_t source_rows = max_rows < num_src_rows ? max_rows : num_src_rows;  // that can be read
        while (((max_rows * row_bytes) >> group_log2) > kPackGroupBytes * (group_log2 < 5 ? group_log2 : 6) / 3 ||
               ((source_rows * row_bytes) >> group_log2) > kPackSourceBytes)
            if (++group_log2 == 16) break;
        // rounding down the parts of every rank's list can put one more row per rank into a group
        const int64_t needed = ((max_rows + (int64_t(1) << group_log2) - 1) >> group_log2) + num_ranks;
        const uint32_t slots = uint32_t(needed < (1 << 14) ? needed : (1 << 14));  // the kernel goes round for the rest
        const unsigned blocks = slots << group_log2;
        if (stream_rows)
            launch(pack_groups_kernel<true>, blocks, threads, 0, hs, send_cumsum, sorted_token_ids, max_rows, num_ranks,
                                                                 group_log2, slots, a);
        else
            launch(pack_groups_kernel<false>, blocks, threads, 0, hs, send_cumsum, sorted_token_ids, max_rows, num_ranks,
                                                                  group_log2, slots, a);
    } else {
        const unsigned blocks = unsigned(max_rows < (int64_t(1) << 22) ? max_rows : int64_t(1) << 22);
        if (stream_rows)
            launch(pack_rows_kernel<true>, blocks, threads, 0, hs, num_rows_dev, sorted_token_ids, max_rows, blocks, a);
        else
            launch(pack_rows_kernel<false>, blocks, threads, 0, hs, num_rows_dev, sorted_token_ids, max_rows, blocks, a);
    }
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_pack_rows(const void* src, const void* scale_src, const int64_t* sorted_token_ids,
                     const int64_t* num_rows_dev, int64_t max_rows, int num_src_rows, int row_bytes,
                     int scale_row_bytes, void* dst, void* scale_dst, void* stream) {
    return deepep_pack_rows_by_rank(src, scale_src, sorted_token_ids, num_rows_dev, nullptr, 0, max_rows, num_src_rows,
                                    row_bytes, scale_row_bytes, dst, scale_dst, stream);
}

}  // extern "C"
