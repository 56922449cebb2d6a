// What a rank derives from the gathered route counts before the exchange of a
// low-latency dispatch: rows to send to and to expect from every rank, where its
// returned rows start inside every peer's combine buffer, and one metadata
// record per row it will receive.  The reference computes all of it on the host
// from three device-to-host copies (csrc/transport/ll_pipeline.cpp:1204-1269 and
// :1277-1361); here it is one launch on the stream the counts arrive on.
#include "common.hpp"
#include "../../include/deepep_hip.h"

namespace deepep {

constexpr int kExchangeThreads = 256, kExchangeWaves = kExchangeThreads / kWave;
constexpr int kExchangeMaxRanks = 1024;

// Sum over the wave of 64-bit values below 2^48, in two parts whose sums fit 32 bits (DPP, no LDS).
__device__ __forceinline__ int64_t wave_sum_u48(int64_t v) {
    const uint32_t low = __builtin_amdgcn_readlane(wave_inclusive_sum(int(v & 0xffffff)), kWave - 1);
    const uint32_t high = __builtin_amdgcn_readlane(wave_inclusive_sum(int(v >> 24)), kWave - 1);
    return (int64_t(high) << 24) + low;
}

// The first workgroup writes the per-rank outputs, the next ones a source rank a wave (what it sent to the ranks below this
// one), the others the row records; whether a count is out of bounds, and the prefix of the rows expected from each rank,
// the first and the last derive themselves, from L2.  Instructions bound it: a count that only has to be checked is one
// maximum, four to a load, all loads go out ahead of the first wait, and workgroups have four waves, one for each SIMD of a
// compute unit.  Sixteen waves that summed every row in every workgroup / this, microseconds in a row: 8 ranks x 64 experts
// 3.2 / 2.8, 16 x 128 3.7 / 2.8, 32 x 256 4.6 / 2.9, 64 x 1024 11.4 / 7.0, 1024 x 1024 178 / 84.
__global__ __launch_bounds__(kExchangeThreads) void ll_exchange_meta_kernel(
    const int32_t* __restrict__ all_num_routed, int num_experts, int num_ranks, int rank, int max_tokens,
    int64_t row_capacity, int32_t* __restrict__ send_counts, int32_t* __restrict__ recv_counts,
    int32_t* __restrict__ totals, int64_t* __restrict__ combine_remote_recv_offset,
    uint32_t* __restrict__ source_rank, uint32_t* __restrict__ source_offset, uint32_t* __restrict__ padded_index,
    uint32_t* __restrict__ combine_send_offset, uint32_t* __restrict__ num_recv_tokens,
    uint32_t* __restrict__ tokens_per_expert) {
    __shared__ int32_t recv_prefix[kExchangeMaxRanks + 1];
    __shared__ int32_t recv_of[kExchangeMaxRanks];
    __shared__ int32_t send_to[kExchangeMaxRanks];  // the first workgroup's
    __shared__ uint32_t wave_found[kExchangeWaves];
    const int tid = threadIdx.x, lane = lane_id(), w = wave_in_block();
    const uint32_t experts_per_rank = uint32_t(num_experts / num_ranks), first_expert = rank * experts_per_rank;
    const int row_blocks = (num_ranks + kExchangeWaves - 1) / kExchangeWaves;
    const bool writes_totals = blockIdx.x == 0;
    if (!writes_totals && int(blockIdx.x) <= row_blocks) {
        // where this rank's returned rows start in the peer's combine buffer: behind what the peer
        // sent to the ranks below this one (csrc/transport/ll_pipeline.cpp:1283-1295, computed
        // from the raw counts whatever their state)
        const int peer = int(blockIdx.x - 1) * kExchangeWaves + w;
        if (peer >= num_ranks) return;
        const int32_t* row = all_num_routed + int64_t(peer) * num_experts;
        int64_t below = 0;
        for (uint32_t e0 = 0; e0 < first_expert; e0 += 4 * kWave) {
            uint32_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t e = e0 + u * kWave + lane;
                v[u] = uint32_t(row[e < first_expert ? e : 0]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) below += e0 + u * kWave + lane < first_expert ? int64_t(v[u]) : 0;
        }
        below = wave_sum_u48(below);
        if (lane == 0) combine_remote_recv_offset[peer] = below;
        return;
    }
    // ---- the first loads of everything, before anything waits ----------------
    constexpr int kAhead = 8, kPass = kAhead * kExchangeThreads * 4;  // counts
    const int64_t n = int64_t(num_ranks) * num_experts;
    const auto pass_at = [&](int64_t base) {  // zeros past the last count
        return row_buffer(reinterpret_cast<const uint8_t*>(all_num_routed + base), int(n - base < kPass ? n - base : kPass) * 4);
    };
    u32x4 v[kAhead];
    {
        const auto counts = pass_at(0);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = load_row_u32x4<false>(counts, (u * kExchangeThreads + tid) * 16);
    }
    // entry i of what every rank sends to this one, rank by rank
    const auto to_me = [&](uint32_t i) {
        const uint32_t r = i / experts_per_rank;
        return all_num_routed + int64_t(r) * num_experts + first_expert + (i - r * experts_per_rank);
    };
    const int32_t* mine = all_num_routed + int64_t(rank) * num_experts;
    const uint32_t experts = uint32_t(num_experts), i0 = uint32_t(tid) < experts ? tid : 0;
    const int received = *to_me(i0), sent = mine[i0];
    for (int r = tid; r < num_ranks; r += kExchangeThreads) recv_of[r] = send_to[r] = 0;
    lds_barrier();

    // a count above the per-expert bound marks the whole gather as corrupt: nobody sends or
    // receives this time (csrc/transport/ll_pipeline.cpp:1216-1248)
    const uint32_t max_per_expert = max_tokens > 0 ? uint32_t(max_tokens) : 4096u;
    uint32_t most = 0;
    for (int64_t base = 0;;) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) most = most > v[u][i] ? most : v[u][i];
        base += kPass;
        if (base >= n) break;
        const auto counts = pass_at(base);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = load_row_u32x4<false>(counts, (u * kExchangeThreads + tid) * 16);
    }
    const uint64_t bad = __ballot(most > max_per_expert);
    if (lane == 0) wave_found[w] = bad != 0 ? 1u : 0u;
    // Lanes of one rank would wait for one another at its word: where a wave's are all of one, it hands in their sum (8 ranks x
    // 1024 experts 4.3 -> 3.8 us, 8 x 4096 10.9 -> 9.7).
    const bool waves_of_one_rank = experts_per_rank % kWave == 0;
    const auto add = [&](int32_t* to, uint32_t i, int count) {
        if (waves_of_one_rank) {
            count = wave_inclusive_sum(count);
            if (lane != kWave - 1) return;
        }
        atomicAdd(&to[i / experts_per_rank], count);
    };
    if (uint32_t(tid) < experts) {
        add(recv_of, tid, received);
        if (writes_totals) add(send_to, tid, sent);
    }
    for (uint32_t i = tid + kExchangeThreads; i < experts; i += kExchangeThreads) {
        add(recv_of, i, *to_me(i));
        if (writes_totals) add(send_to, i, mine[i]);
    }
    lds_barrier();
    bool is_corrupt = false;
#pragma unroll
    for (int i = 0; i < kExchangeWaves; ++i) is_corrupt |= wave_found[i] != 0;

    if (tid < kWave) {  // exclusive prefix over the ranks, one wave
        int carry = 0;
        for (int r0 = 0; r0 < num_ranks; r0 += kWave) {
            const int r = r0 + tid;
            const int of = r < num_ranks && !is_corrupt ? recv_of[r] : 0;
            const int inc = wave_inclusive_sum(of);
            if (r < num_ranks) recv_prefix[r] = carry + inc - of;
            carry += __builtin_amdgcn_readlane(inc, kWave - 1);
        }
        if (tid == 0) recv_prefix[num_ranks] = carry;
    }
    lds_barrier();
    int total_recv = recv_prefix[num_ranks];
    const int all_expected = total_recv;
    // csrc/transport/ll_pipeline.cpp:1306-1312: an impossible total receives nothing
    const int64_t max_possible = int64_t(num_ranks) * max_tokens * 8;
    int64_t rows = total_recv;
    if (rows < 0 || rows > max_possible) rows = 0, total_recv = 0;
    if (rows > row_capacity) rows = row_capacity;

    if (writes_totals) {
        for (int r = tid; r < num_ranks; r += kExchangeThreads) {
            send_counts[r] = is_corrupt ? 0 : send_to[r];
            recv_counts[r] = is_corrupt ? 0 : recv_of[r];
        }
        for (uint32_t e = tid; e < experts_per_rank; e += kExchangeThreads) tokens_per_expert[e] = 0;
        if (w == 1) {  // total sent
            int part = 0;
            if (!is_corrupt)
                for (int r = lane; r < num_ranks; r += kWave) part += send_to[r];
            const int total_send = __builtin_amdgcn_readlane(wave_inclusive_sum(part), kWave - 1);
            if (lane == 0) totals[0] = total_send, totals[1] = all_expected, totals[2] = is_corrupt ? 1 : 0;
        }
        if (tid == 0) num_recv_tokens[0] = uint32_t(total_recv), num_recv_tokens[1] = uint32_t(rows);
        return;
    }
    // one record per expected row, grouped by source rank (csrc/transport/ll_pipeline.cpp:1319-1343)
    const int record_blocks = int(gridDim.x) - 1 - row_blocks;
    for (int64_t i = int64_t(int(blockIdx.x) - 1 - row_blocks) * kExchangeThreads + tid; i < rows;
         i += int64_t(record_blocks) * kExchangeThreads) {
        int lo = 0, hi = num_ranks;  // recv_prefix[lo] <= i < recv_prefix[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (recv_prefix[mid] <= i) lo = mid; else hi = mid;
        }
        const uint32_t t = uint32_t(i - recv_prefix[lo]);
        source_rank[i] = uint32_t(lo);
        source_offset[i] = uint32_t(lo) * uint32_t(max_tokens) + t;
        padded_index[i] = uint32_t(i);
        combine_send_offset[i] = uint32_t(recv_prefix[lo]) + t;
    }
}

}  // namespace deepep

using namespace deepep;

extern "C" int deepep_ll_exchange_metadata(const int32_t* all_num_routed, int num_experts, int num_ranks, int rank,
                                           int num_max_dispatch_tokens_per_rank, int64_t row_capacity,
                                           int32_t* send_counts, int32_t* recv_counts, int32_t* totals,
                                           int64_t* combine_remote_recv_offset, uint32_t* source_rank,
                                           uint32_t* source_offset, uint32_t* padded_index,
                                           uint32_t* combine_send_offset, uint32_t* num_recv_tokens,
                                           uint32_t* tokens_per_expert, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_ranks > 0 && num_ranks <= kExchangeMaxRanks);
    EP_HOST_ASSERT(num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(rank >= 0 && rank < num_ranks);
    EP_HOST_ASSERT(int64_t(num_ranks) * num_experts < (int64_t(1) << 30));
    EP_HOST_ASSERT(row_capacity >= 0 && row_capacity < (int64_t(1) << 32));
    EP_HOST_ASSERT(all_num_routed != nullptr && send_counts != nullptr && recv_counts != nullptr && totals != nullptr);
    EP_HOST_ASSERT(combine_remote_recv_offset != nullptr && num_recv_tokens != nullptr && tokens_per_expert != nullptr);
    EP_HOST_ASSERT(row_capacity == 0 || (source_rank != nullptr && source_offset != nullptr &&
                                         padded_index != nullptr && combine_send_offset != nullptr));
    // Workgroups for the records, one after another for a thread: 8 ranks x 256 experts, 3800 rows of 4096 4.4 -> 5.1 us with
    // eight a thread, 8 x 64, 256000 of 300000 5.3 -> 7.8 with 64 workgroups.
    int64_t records = (row_capacity + 4 * kExchangeThreads - 1) / (4 * kExchangeThreads);
    records = records > 256 ? 256 : records;
    const int64_t blocks = 1 + (num_ranks + kExchangeWaves - 1) / kExchangeWaves + records;
    launch(ll_exchange_meta_kernel, unsigned(blocks), kExchangeThreads, 0, reinterpret_cast<hipStream_t>(stream),
        all_num_routed, num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank, row_capacity, send_counts,
        recv_counts, totals, combine_remote_recv_offset, source_rank, source_offset, padded_index,
        combine_send_offset, num_recv_tokens, tokens_per_expert);
    EP_LAUNCH_CHECK();
    return 0;
}
