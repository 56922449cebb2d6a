// Helpers for kernels that walk a list of variable-length row segments with
// one wavefront per row (part): the segment prefix held in a wave's registers
// with its row -> segment lookup, a workgroup-wide exclusive scan in LDS for the
// metadata pass, the 16-byte-per-lane row copy, and the index + flat-copy pair
// of kernels for large batches.
#pragma once

#include "common.hpp"

namespace deepep {

// ---------------------------------------------------------------------
// Exclusive prefix of n ints held in LDS, by the whole workgroup (a multiple
// of 64 threads, at most 1024).  data[n] receives the total; wave_totals has
// room for 16 ints.
// ---------------------------------------------------------------------
constexpr int kMaxBlockWaves = 16;

__device__ __forceinline__ void block_exclusive_scan(int32_t* data, int n, int32_t* wave_totals) {
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const int threads = block_threads(), waves = threads >> 6;
    const int per = (n + threads - 1) / threads;
    const int lo = tid * per;
    int sum = 0;
    for (int j = 0; j < per; ++j)
        if (lo + j < n) sum += data[lo + j];
    const int incl = wave_inclusive_sum(sum);
    if (lane == kWave - 1) wave_totals[w] = incl;
    lds_barrier();
    int offset = incl - sum, total = 0;
    for (int w2 = 0; w2 < waves; ++w2) {
        const int t = wave_totals[w2];
        if (w2 < w) offset += t;
        total += t;
    }
    int run = offset;
    for (int j = 0; j < per; ++j)
        if (lo + j < n) {
            const int v = data[lo + j];
            data[lo + j] = run;
            run += v;
        }
    if (tid == 0) data[n] = total;
    lds_barrier();
}

// ---------------------------------------------------------------------
// The same prefix, held by one wave in registers: no LDS and no barrier, so a
// wave can start looking up rows as soon as its own loads of the counts are
// back.  Lane l holds the counts of segments [l * kPer, (l + 1) * kPer) and the
// number of rows in all lower lanes' segments.  kPer is a compile-time 4 (up to
// 256 segments) or 16 (up to 1024) so that every index below is static and the
// arrays stay in registers.
// ---------------------------------------------------------------------
template <int kPer>
struct WaveSegments {
    int cnt[kPer];
    int aux[kPer];  // one caller-defined value per segment, returned by the lookup
    int lane_base;  // rows in the segments held by lower lanes
    int total;      // rows in all segments
};

// Lane l's kPer consecutive values p[l * kPer + u] (0 beyond n), as 16-byte loads where a whole
// vector lies inside the array.  p must be 16-byte aligned.  Arrays of whole vectors are read as a
// buffer, whose loads past the end give zeros without a branch for each of them.
template <int kPer>
__device__ __forceinline__ void wave_load_int32(const int32_t* __restrict__ p, int n, int lane, int (&out)[kPer]) {
    static_assert(kPer % 4 == 0, "whole 16-byte vectors per lane");
    if (n % 4 == 0) {
        const auto all = row_buffer(reinterpret_cast<const uint8_t*>(p), n * 4);
#pragma unroll
        for (int v = 0; v < kPer / 4; ++v) {
            const u32x4 q = load_row_u32x4<false>(all, lane * kPer * 4 + v * 16);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[v * 4 + i] = int(q[i]);
        }
        return;
    }
#pragma unroll
    for (int v = 0; v < kPer / 4; ++v) {
        const int s0 = lane * kPer + v * 4;
        if (s0 + 3 < n) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(p + s0);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[v * 4 + i] = int(q[i]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) out[v * 4 + i] = s0 + i < n ? p[s0 + i] : 0;
        }
    }
}

template <int kPer>
__device__ __forceinline__ void wave_load_int64(const int64_t* __restrict__ p, int n, int lane,
                                                int64_t (&out)[kPer]) {
    static_assert(kPer % 2 == 0, "whole 16-byte vectors per lane");
    if (n % 2 == 0) {
        const auto all = row_buffer(reinterpret_cast<const uint8_t*>(p), n * 8);
#pragma unroll
        for (int v = 0; v < kPer / 2; ++v) {
            const u32x4 q = load_row_u32x4<false>(all, lane * kPer * 8 + v * 16);
            out[v * 2] = int64_t((uint64_t(q[1]) << 32) | q[0]);
            out[v * 2 + 1] = int64_t((uint64_t(q[3]) << 32) | q[2]);
        }
        return;
    }
#pragma unroll
    for (int v = 0; v < kPer / 2; ++v) {
        const int s0 = lane * kPer + v * 2;
        if (s0 + 1 < n) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(p + s0);
            out[v * 2] = int64_t((uint64_t(q[1]) << 32) | q[0]);
            out[v * 2 + 1] = int64_t((uint64_t(q[3]) << 32) | q[2]);
        } else {
            out[v * 2] = s0 < n ? p[s0] : 0;
            out[v * 2 + 1] = 0;
        }
    }
}

// Finishes a table whose cnt[] the caller has filled (zero beyond the last segment).
template <int kPer>
__device__ __forceinline__ void wave_segments_finish(WaveSegments<kPer>& t) {
    int mine = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) mine += t.cnt[u];
    const int incl = wave_inclusive_sum(mine);
    t.lane_base = incl - mine;
    t.total = __builtin_amdgcn_readlane(incl, kWave - 1);
}

// Rows before segment q (wave-uniform q in [0, 64 * kPer]).
template <int kPer>
__device__ __forceinline__ int wave_segments_prefix(const WaveSegments<kPer>& t, int q) {
    q = __builtin_amdgcn_readfirstlane(q);
    const int owner = q / kPer, within = q % kPer;
    if (owner >= kWave) return t.total;
    int run = t.lane_base;
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (u < within) run += t.cnt[u];
    return __builtin_amdgcn_readlane(run, owner);
}

// Segment holding row (wave-uniform, 0 <= row < total); seg_first receives the rows before it,
// seg_aux the segment's aux value.
template <int kPer>
__device__ __forceinline__ int wave_segments_find(const WaveSegments<kPer>& t, int row, int& seg_first,
                                                  int& seg_aux) {
    // the last lane whose base is <= row owns the row (empty lanes share their successor's base)
    const int owner = __builtin_amdgcn_readfirstlane(__popcll(__ballot(t.lane_base <= row)) - 1);
    int run = t.lane_base, found = 0, first = t.lane_base, aux = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        if (run <= row && row < run + t.cnt[u]) found = u, first = run, aux = t.aux[u];
        run += t.cnt[u];
    }
    seg_first = __builtin_amdgcn_readlane(first, owner);
    seg_aux = __builtin_amdgcn_readlane(aux, owner);
    return owner * kPer + __builtin_amdgcn_readlane(found, owner);
}

// Segments, in (expert, source) order, to experts: n / num_ranks for n below 2^16 by one multiplication.
struct RankDivider {
    uint32_t magic;  // 0: one rank
    __device__ __forceinline__ int operator()(int n) const { return magic != 0 ? int(__umulhi(uint32_t(n), magic)) : n; }
};
inline RankDivider make_rank_divider(int num_ranks) {
    return RankDivider{num_ranks == 1 ? 0u : uint32_t(((uint64_t(1) << 32) + num_ranks - 1) / num_ranks)};
}

// A row of num_vec vectors cut into 2^parts_log2 runs of whole 64-vector (1 KiB) chunks.
__device__ __forceinline__ void row_part_range(int num_vec, int parts_log2, int part, int& v_begin, int& v_end) {
    const int chunks = (num_vec + kWave - 1) / kWave;
    const int per = (chunks + (1 << parts_log2) - 1) >> parts_log2;
    v_begin = min(part * per * kWave, num_vec);
    v_end = min(v_begin + per * kWave, num_vec);
}

// Vectors [v_begin, v_end) of a row, moved by one wave, kDepth KiB of it in flight: the first of them in `r` between
// load() and store(), which moves the others too.
template <int kDepth, bool kStreamLoad, bool kStreamStore>
struct RowPart {
    u32x4 r[kDepth];
    const uint8_t* src;
    int bytes;
    __device__ __forceinline__ void load(const uint8_t* row, int v_begin, int v_end, int lane) {
        src = row + v_begin * 16, bytes = (v_end - v_begin) * 16;
        const auto from = row_buffer(src, bytes);
#pragma unroll
        for (int u = 0; u < kDepth; ++u) r[u] = load_row_u32x4<kStreamLoad>(from, lane * 16 + u * 1024);
    }
    __device__ __forceinline__ void store(uint8_t* row, int v_begin, int lane) {
        const auto from = row_buffer(src, bytes), to = row_buffer(row + v_begin * 16, bytes);
        for (int base = lane * 16;;) {
#pragma unroll
            for (int u = 0; u < kDepth; ++u) store_row_u32x4<kStreamStore>(to, base + u * 1024, r[u]);
            base += kDepth * 1024;
            if (base - lane * 16 >= bytes) return;
#pragma unroll
            for (int u = 0; u < kDepth; ++u) r[u] = load_row_u32x4<kStreamLoad>(from, base + u * 1024);
        }
    }
};

// Host-side choice of the row split (log2 of the parts): small problems cannot fill the chip with one wave per row, and
// in larger ones a wave that takes a whole row is what the launch ends up waiting for.  Microseconds of a dispatch and a
// combine in one launch, rows whole / in parts: 8800 rows of 14 KB 112.5 / 109.4, 10400 of 8 KB 82.2 / 80.8, 14400 of 4 KB
// 61.6 / 60.8, 21600 of 4 KB 85.2 / 82.8, 28000 of 4 KB 103.1 / 100.8, but of 3 KB 84.0 / 85.0, 32768 of 2 KB 69.4 / 71.5.
// Past 8192 rows not those of less than 4 KB, nor past 256 segments, where finding a row's place costs four times as much.
// The combine alone: 12000 rows of 256 bytes 6.5 / 9.6, of 1 KB 8.6 / 12.2, of 2 KB 12.4 / 15.0, of 3 KB 17.8 / 18.2, of 4 KB
// 23.3 / 22.8; 8240 rows from 1024 experts of 256 bytes 13.0 / 21.9, of 4 KB 19.9 / 26.2, of 14 KB 61.5 / 68.1.
inline int choose_row_parts_log2(int64_t estimated_rows, int64_t row_bytes, int num_segments) {
    if (estimated_rows > 8192 && (row_bytes < 4096 || num_segments > 4 * kWave || estimated_rows > 32768)) return 0;
    return row_bytes > 8192 ? 2 : 1;
}

// ---------------------------------------------------------------------
// Large batches.  A flat copy — one workgroup per row, one 16-byte vector per
// thread, no loop — is what reaches the highest HBM rate on this GPU, but it
// needs the row -> (source, destination) map up front.  ll_segment_index_kernel
// builds it: one workgroup per segment scans the segment counts (<= 1024 ints)
// and writes a descriptor {source row, destination row} for each of its rows.
// ---------------------------------------------------------------------
struct RowDesc {
    int32_t src_row;  // row index in the source buffer; < 0: nothing to copy
    int32_t dst_row;  // >= 0: row index in the primary destination; < 0: -(1 + row) in the secondary one
};

// Where a dispatch reports the rows it received to a host that sizes the next one by it: (tokens sent << 32) | rows,
// one 8-byte store into pinned memory that the host reads whenever it likes.  A null word reports nothing.
struct ObservedRows {
    uint64_t* host;
    uint32_t tokens;
};
__device__ __forceinline__ void report_observed(const ObservedRows& o, int rows) {
    if (o.host != nullptr)
        __hip_atomic_store(o.host, (uint64_t(o.tokens) << 32) | uint32_t(rows), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kIndexThreads = 1024;

// Exclusive prefix over one value per thread of a 1024-thread workgroup; returns the prefix, sets total.
__device__ __forceinline__ int block_exclusive_scan_1024(int v, int32_t* wave_totals, int& total) {
    const int lane = lane_id(), w = int(threadIdx.x) >> 6;
    const int incl = wave_inclusive_sum(v);
    if (lane == kWave - 1) wave_totals[w] = incl;
    __syncthreads();
    int offset = incl - v;
    total = 0;
    for (int w2 = 0; w2 < kIndexThreads / kWave; ++w2) {
        const int t = wave_totals[w2];
        if (w2 < w) offset += t;
        total += t;
    }
    return offset;
}

// Dispatch receive: counts = recv_count; writes layout_range / packed_count / stats;
// descriptor = {staging row seg*M + j, packed row e_l*N + begin + j}; rank = -1, or the rank
// whose own rows the send side has already put at their packed position (they keep their
// place in the ranges, in ascending source order, and get no descriptors).
static __global__ __launch_bounds__(kIndexThreads) void ll_segment_index_kernel(
    const int32_t* __restrict__ counts32, int num_local_experts, int num_ranks, int rank, int max_tokens,
    int64_t* __restrict__ layout_out, int32_t* __restrict__ packed_count, int32_t* __restrict__ stats,
    int32_t* __restrict__ flat_out, RowDesc* __restrict__ desc, ObservedRows observed) {
    __shared__ int32_t flat[kIndexThreads + 1];   // prefix over the rows that get descriptors
    __shared__ int32_t place[kIndexThreads + 1];  // prefix over all rows: where a segment lands
    __shared__ int32_t wave_totals[kIndexThreads / kWave];
    __shared__ int32_t wave_totals_place[kIndexThreads / kWave];
    const int tid = threadIdx.x;
    const int num_segments = num_local_experts * num_ranks;
    int c = 0;
    if (tid < num_segments) {
        c = counts32[tid];
        c = c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
    }
    // rank >= 0: the rank's own rows are already in place (reference order: a range
    // begins where the lower source ranks' rows end, csrc/kernels/efa_kernels.cu:991-1010), so
    // they count towards where the later segments land but take no descriptors
    const bool own_placed = rank >= 0;
    const int c_all = c;
    if (own_placed && tid < num_segments && tid % num_ranks == rank) c = 0;
    int total;
    const int prefix = block_exclusive_scan_1024(c, wave_totals, total);
    if (tid < num_segments) flat[tid] = prefix;
    if (tid == 0) flat[num_segments] = total;
    int total_all = total, prefix_all = prefix;
    if (own_placed) prefix_all = block_exclusive_scan_1024(c_all, wave_totals_place, total_all);
    if (tid < num_segments) place[tid] = prefix_all;
    if (tid == 0) place[num_segments] = total_all;
    __syncthreads();
    const int64_t slots_per_expert = int64_t(max_tokens) * num_ranks;
    if (blockIdx.x == 0) {
        for (int s = tid; s <= num_segments; s += kIndexThreads) flat_out[s] = flat[s];
        if (tid == 0) report_observed(observed, place[num_segments]);
        if (tid < num_segments) {
            const int le = tid / num_ranks;
            const int64_t cnt = c_all;
            const int64_t begin = place[tid] - place[le * num_ranks];
            layout_out[tid] = cnt > 0 ? ((begin << 32) | cnt) : 0;
        }
        if (tid < num_local_experts) {
            const int n = place[(tid + 1) * num_ranks] - place[tid * num_ranks];
            packed_count[tid] = n;
            if (stats != nullptr) stats[tid] += n;
        }
    }
    const int seg = blockIdx.x;
    const int le = seg / num_ranks;
    const int cnt = flat[seg + 1] - flat[seg];
    const int64_t begin = place[seg] - place[le * num_ranks];
    for (int j = tid; j < cnt; j += kIndexThreads) {
        RowDesc d;
        d.src_row = seg * max_tokens + j;
        d.dst_row = int32_t(le * slots_per_expert + begin + j);
        desc[flat[seg] + j] = d;
    }
}

// The dispatch-receive index (the kernel above with the rank's own rows already placed) as one workgroup's
// share inside another launch: the send kernel of a large one-call dispatch carries these workgroups
// beside its own, so the index costs no launch.  The launch that carries it is still writing the
// rank's own counts into recv_count, so they are taken from what that launch reads them from: the
// column sums of the per-chunk expert histograms.  Any workgroup size that is a multiple of 64;
// lds holds 2 * (segments + 1) ints, wave_totals 16.
struct FusedIndexArgs {
    const int32_t* recv_count;  // [E_l][R]; the own column is not read
    const int32_t* chunk_hist;  // [chunks][E] of this rank's own entries
    int num_chunks, num_experts, num_local_experts, num_ranks, rank, max_tokens;
    int64_t* layout_out;
    int32_t* packed_count;
    int32_t* stats;
    int32_t* flat_out;
    RowDesc* desc;
    ObservedRows observed;
};

__device__ __forceinline__ void recv_index_block(const FusedIndexArgs& a, int seg, int32_t* lds, int32_t* wave_totals) {
    const int tid = threadIdx.x, threads = block_threads();
    const int num_ranks = a.num_ranks, max_tokens = a.max_tokens;
    const int num_segments = a.num_local_experts * num_ranks;
    int32_t* flat = lds;                      // prefix over the rows that get descriptors
    int32_t* place = lds + num_segments + 1;  // prefix over all rows: where a segment lands
    for (int s = tid; s < num_segments; s += threads) {
        const int le = s / num_ranks, src = s - le * num_ranks;
        int c = 0;
        if (src == a.rank) {
            const int e = a.rank * a.num_local_experts + le;
            for (int c0 = 0; c0 < a.num_chunks; c0 += 8) {  // eight loads in flight
                int v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    v[u] = c0 + u < a.num_chunks ? a.chunk_hist[int64_t(c0 + u) * a.num_experts + e] : 0;
#pragma unroll
                for (int u = 0; u < 8; ++u) c += v[u];
            }
        } else {
            c = a.recv_count[s];
        }
        c = c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
        place[s] = c;
        flat[s] = src == a.rank ? 0 : c;  // own rows are in place already: no descriptors
    }
    lds_barrier();
    block_exclusive_scan(flat, num_segments, wave_totals);
    block_exclusive_scan(place, num_segments, wave_totals);
    const int64_t slots_per_expert = int64_t(max_tokens) * num_ranks;
    if (seg == 0) {
        if (tid == 0) report_observed(a.observed, place[num_segments]);
        for (int s = tid; s <= num_segments; s += threads) a.flat_out[s] = flat[s];
        for (int s = tid; s < num_segments; s += threads) {
            const int le = s / num_ranks;
            const int64_t cnt = place[s + 1] - place[s];
            const int64_t begin = place[s] - place[le * num_ranks];
            a.layout_out[s] = cnt > 0 ? ((begin << 32) | cnt) : 0;
        }
        for (int le = tid; le < a.num_local_experts; le += threads) {
            const int n = place[(le + 1) * num_ranks] - place[le * num_ranks];
            a.packed_count[le] = n;
            if (a.stats != nullptr) a.stats[le] += n;
        }
    }
    const int le = seg / num_ranks;
    const int cnt = flat[seg + 1] - flat[seg];
    const int64_t begin = place[seg] - place[le * num_ranks];
    for (int j = tid; j < cnt; j += threads) {
        RowDesc d;
        d.src_row = seg * max_tokens + j;
        d.dst_row = int32_t(le * slots_per_expert + begin + j);
        a.desc[flat[seg] + j] = d;
    }
}

// The index of the combine's row return: counts and begins from layout_range; descriptor = {expert-output row
// e_l*N + begin + j, seg*M + j for other ranks or -(1 + (rank*E_l + e_l)*M + j) for this rank's own rows}.  One
// workgroup's share: of a launch of its own or, in front of the reduce's workgroups, of the reduce's launch.
// Any workgroup size that is a multiple of 64; lds holds segments + 1 ints, wave_totals 16.
struct CombineIndexArgs {
    const int64_t* layout_range;  // [E_l][R]
    int num_local_experts, num_ranks, rank, max_tokens;
    bool skip_own;  // own rows stay where they are
    int32_t* flat_out;
    RowDesc* desc;
};

__device__ __forceinline__ void combine_index_block(const CombineIndexArgs& a, int seg, int32_t* flat,
                                                    int32_t* wave_totals) {
    const int tid = threadIdx.x, threads = block_threads();
    const int num_ranks = a.num_ranks, max_tokens = a.max_tokens;
    const int num_segments = a.num_local_experts * num_ranks;
    const int64_t begin = a.layout_range[seg] >> 32;
    for (int s = tid; s < num_segments; s += threads) {
        const int c = int(a.layout_range[s] & 0xffffffffll);
        flat[s] = c < 0 || (a.skip_own && s % num_ranks == a.rank) ? 0 : (c > max_tokens ? max_tokens : c);
    }
    lds_barrier();
    block_exclusive_scan(flat, num_segments, wave_totals);
    if (seg == 0)
        for (int s = tid; s <= num_segments; s += threads) a.flat_out[s] = flat[s];
    const int le = seg / num_ranks, s = seg - le * num_ranks;
    const int first = flat[seg], cnt = flat[seg + 1] - first;
    const int64_t slots_per_expert = int64_t(max_tokens) * num_ranks;
    const bool sound = begin >= 0 && begin + cnt <= slots_per_expert;  // rows of a malformed range are not moved
    for (int j = tid; j < cnt; j += threads) {
        RowDesc d;
        d.src_row = sound ? int32_t(le * slots_per_expert + begin + j) : -1;
        d.dst_row = s == a.rank ? -(1 + (a.rank * a.num_local_experts + le) * max_tokens + j) : seg * max_tokens + j;
        a.desc[first + j] = d;
    }
}

// One workgroup per described row (looping only if there are more rows than workgroups).  Only batches too large for
// the caches come here, so the payload streams, one 16-byte vector a thread: two workgroups of a 14336-byte row are
// what a compute unit holds, and with as few rows as that in flight HBM serves them best, provided that a row's
// address is there early.  Hence two trips to memory in front of the row and no more (the arguments; then descriptor and
// number of rows together: left to the compiler it is four), buffer addressing, and no row that waits for another one.
// Beyond a few hundred MB address translation bounds it as well, which likes the rows in flight to be close together:
// workgroup i runs on XCD i % 8, and each XCD is given kFlatWindow rows in a row instead of every eighth one.
// Microseconds against two vectors a thread, four trips and a grid of one workgroup for two rows:
//   28672 rows of 14336 bytes 131.3 -> 125.5 (6.55 TB/s), 7168 bytes and scales 67.8 -> 65.7;
//   160000 of 14336 bytes 792 -> 712 (6.5 TB/s), 14300 of 7168 41.5 -> 39.8.
// A bare copy of whole rows, nothing in front of it, reaches 6.7.  Workgroups that loop are slower however early they
// fetch what comes next: 32768 x 14336 bytes 142.5 us with a row each, 145 with two, 153 with four, 164 with eight,
// 165 to 175 with 512 workgroups that stay.
constexpr int kFlatWindow = 32;
constexpr int kFlatRound = 8 * kFlatWindow;

__device__ __forceinline__ uint32_t flat_row_of_block(uint32_t block) {
    const uint32_t in_round = block % kFlatRound;
    return block - in_round + in_round % 8 * kFlatWindow + in_round / 8;
}
__device__ __forceinline__ uint32_t flat_rounds_end(uint32_t rows) {
    return (rows + kFlatRound - 1) / kFlatRound * kFlatRound;
}

// What a row carries besides its payload (the dispatch's rows; all null for the combine's).
struct FlatTails {
    uint8_t* scale_dst;
    int32_t* src_info;
    uint32_t scale_dwords, scale_off, info_off;
};

template <bool kTails>
static __global__ __launch_bounds__(1024) void ll_rows_flat_kernel(
    const int32_t* __restrict__ total, const RowDesc* __restrict__ desc, uint32_t capacity, uint32_t grid,
    const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t src_stride, uint32_t dst_stride, int num_vec,
    int data_threads, uint8_t* __restrict__ dst_own, FlatTails tails) {
    const int tid = threadIdx.x;
    uint32_t i = blockIdx.x, row = flat_row_of_block(i);
    // the descriptor is fetched with the number of rows, not behind it: the table has `capacity` of them
    const RowDesc* at = desc + (row < capacity ? row : capacity - 1);
    uint32_t rows = uint32_t(*total), src_row = uint32_t(at->src_row), dst_row = uint32_t(at->dst_row);
    await_scalars(rows, src_row, dst_row);
    for (;;) {
        if (row < rows && int32_t(src_row) >= 0) {  // < 0: a record that names no row
            const uint8_t* s = src + uint64_t(src_row) * src_stride;
            if constexpr (kTails) {
                if (wave_in_block() * kWave < data_threads) {
                    block_copy_row<1, true, true>(s, dst + uint64_t(dst_row) * dst_stride, num_vec, tid, data_threads);
                } else {  // the last wave: scales and source index
                    const int lane = lane_id();
                    int32_t info = 0;
                    if (lane == 0) info = *reinterpret_cast<const int32_t*>(s + tails.info_off);
                    const uint32_t* from = reinterpret_cast<const uint32_t*>(s + tails.scale_off);
                    uint32_t* to = reinterpret_cast<uint32_t*>(tails.scale_dst) +
                                   uint64_t(dst_row) * tails.scale_dwords;
                    for (uint32_t v = lane; v < tails.scale_dwords; v += kWave) to[v] = from[v];
                    if (lane == 0) tails.src_info[dst_row] = info;
                }
            } else {
                const bool own = int32_t(dst_row) < 0;
                uint8_t* base = own ? dst_own : dst;
                const uint32_t to = own ? ~dst_row : dst_row;
                if (base != nullptr) block_copy_row<1, true, true>(s, base + uint64_t(to) * dst_stride, num_vec, tid, data_threads);
            }
        }
        if (uint64_t(i) + grid >= flat_rounds_end(rows)) break;
        i += grid, row = flat_row_of_block(i);
        if (row < rows) src_row = uint32_t(desc[row].src_row), dst_row = uint32_t(desc[row].dst_row);
    }
}

__host__ __device__ inline int64_t segment_workspace_bytes(int num_experts, int max_tokens) {
    const int64_t flat_bytes = ((int64_t(num_experts) + 1) * 4 + 255) & ~int64_t(255);
    return flat_bytes + int64_t(num_experts) * max_tokens * int64_t(sizeof(RowDesc));
}

// Estimated rows above this bound take the index + flat-copy pair instead of the single fused kernel.
constexpr int64_t kLargeBatchRows = 8192;

// Rows a call will probably move: the caller's hint or, without one, a guess from the capacity
// (E * M slots, of which a balanced world fills one in 32 at top-8 of 256 experts).  Only the
// choice between equivalent kernels and the grid sizes depend on it.
inline int64_t estimated_rows(int64_t expected_rows, int64_t num_experts, int64_t max_tokens) {
    return expected_rows > 0 ? expected_rows : num_experts * max_tokens / 32;
}

// Workgroups for `rows` expected rows of at most max_rows.  One that finds no row costs what it takes to launch its
// waves, ten to seventeen a nanosecond (for 14336-byte rows 1.45 ns, 7168 bytes and scales 0.47); one that finds a second
// row about 2 us at the very end: a thirty-second more than expected.  A hint that is too large costs more than one that
// is too small by as much.  28672 rows of 14336 bytes, sized for an eighth of them, half, all, twice, eight times: 142, 130,
// 125, 165, 415 us.  No more than a launch takes, which is 2^32 - 1 threads.
inline unsigned flat_grid_blocks(int64_t rows, int64_t max_rows, int threads) {
    int64_t want = rows + rows / 32 + 64;
    if (want > max_rows) want = max_rows;
    if (want > (int64_t(1) << 22)) want = int64_t(1) << 22;
    if (want < 1) want = 1;
    want = (want + kFlatRound - 1) / kFlatRound * kFlatRound;  // whole rounds over the XCDs
    const int64_t most = 0xffffffffll / threads / kFlatRound * kFlatRound;
    return unsigned(want < most ? want : most);
}

// Rows a copy is sized for when only a bound is known: what fits can be a thousand times what comes.  64 workgroups a
// compute unit.  Return by destination of 14336-byte rows with room for a million, us, sized like this / for the room / by
// the rows: 1000 rows 17 / 820 / 5.5, 8192 42 / 847 / 37, 28672 128 / 920 / 127, 160000 789 / 1445 / 758.
constexpr int64_t kFlatRowsUnhinted = 16384;
inline int64_t flat_rows_expected(int64_t expected_rows, int64_t max_rows) {
    return expected_rows > 0 ? expected_rows : (max_rows < kFlatRowsUnhinted ? max_rows : kFlatRowsUnhinted);
}

// The flat copy of the rows `desc` describes (*total of them, memory for max_rows); expected_rows sizes the grid.
inline void launch_rows_flat(const int32_t* total, const RowDesc* desc, int64_t max_rows, int64_t expected_rows,
                             const void* src, int64_t src_stride, int num_vec, void* dst, void* dst_own,
                             int64_t dst_stride, const FlatTails* tails, hipStream_t stream) {
    // Past 65536 rows two a workgroup, while they carry a source index (and scales) and are up to 10 KB.  Microseconds of
    // a skewed dispatch of 166336 rows, one a workgroup / two, in three processes: 2048 bytes 136 to 138 / 126 to 129,
    // 4096 263 to 266 / 243 to 249, 7168 404 to 411 / 397 to 406, bf16 10240 557 to 564 / 538 to 555, but 14336 747 to 755 /
    // 739 to 773; of 83055 rows 74 / 70, 129 / 123, 205 / 207, 284 / 276, 378 / 388.  Without tails below 2 KB (160000
    // rows of 256 bytes 40.2 / 29.6, 512 40.3 / 34.2, 1024 55.8 / 55.7, 1280 74.6 / 69.0); two gain nothing beyond (2048 104.0 /
    // 104.4, 4096 221.5 / 224, 8192 430 / 443, 14336 745 / 753).
    const bool pairs = expected_rows > 65536 && num_vec <= (tails != nullptr ? 640 : 127);
    const int others = tails != nullptr ? kWave : 0, threads = flat_row_threads(num_vec, 1024 - others);
    const unsigned grid = flat_grid_blocks(pairs ? expected_rows / 2 : expected_rows, max_rows, threads + others);
#define DEEPEP_LAUNCH_ROWS(TAILS)                                                                                     \
    launch(ll_rows_flat_kernel<TAILS>, grid, threads + others, 0, stream,                                                 \
        total, desc, uint32_t(max_rows), grid, reinterpret_cast<const uint8_t*>(src), reinterpret_cast<uint8_t*>(dst), \
        uint32_t(src_stride), uint32_t(dst_stride), num_vec, threads, reinterpret_cast<uint8_t*>(dst_own),            \
        tails != nullptr ? *tails : FlatTails{})
    if (tails != nullptr) DEEPEP_LAUNCH_ROWS(true);
    else DEEPEP_LAUNCH_ROWS(false);
#undef DEEPEP_LAUNCH_ROWS
}

}  // namespace deepep
