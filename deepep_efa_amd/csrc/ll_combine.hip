// Low-latency combine: return of the expert outputs (send side) and the
// top-k weighted reduction (receive side).
//
// Data layout in HBM:
//   x (expert outputs)  [E_l][N][H] bf16, live rows given by layout_range
//   combine_staging     [E][M][H] bf16 — slot j of expert e holds the output
//                       for this rank's pair whose dispatch slot was j
//   combine_send_slots  [E_l][R][M][H] bf16 — rows owed to other ranks
#include <algorithm>
#include <cstdlib>

#include "common.hpp"
#include "segments.hpp"
#include "../../include/deepep_hip.h"

namespace deepep {

// ---------------------------------------------------------------------
// Send side: one wave per live row part, rows enumerated segment by segment in
// arrival order (reference: deep_ep/buffer.py:2601-2608 gathers
// x[recv_expert_ids, recv_expert_pos] and un-sorts to arrival order).
// skip_own: the rows owed to this rank itself are left where they are (the
// single-launch combine reads them from x directly).
// ---------------------------------------------------------------------
struct CombineSendArgs {
    const uint8_t* x;
    const int64_t* layout_range;
    int hidden, num_local_experts, num_ranks, rank, max_tokens, parts_log2;
    RankDivider expert_of;
    uint8_t* combine_staging;
    uint8_t* combine_send_slots;
};

// No LDS and no barrier: each wave holds the segment counts and begins in registers.
template <int kPer, bool kStreamLoad, bool kStreamStore>
__device__ __forceinline__ void combine_send_rows_impl(const CombineSendArgs& a, int block, int num_blocks,
                                                       bool skip_own) {
    const int lane = lane_id(), w = wave_in_block();
    const int waves = block_threads() >> 6;
    const int num_ranks = a.num_ranks, max_tokens = a.max_tokens;
    const int num_segments = a.num_local_experts * num_ranks;

    WaveSegments<kPer> seg_table;
    int64_t ranges[kPer];
    DEEPEP_PHASE(0);
    wave_load_int64<kPer>(a.layout_range, num_segments, lane, ranges);
    int source = lane * kPer - a.expert_of(lane * kPer) * num_ranks;  // of segment lane * kPer + u
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        int c = int(ranges[u] & 0xffffffffll);
        c = c < 0 ? 0 : (c > max_tokens ? max_tokens : c);
        if (skip_own && source == a.rank) c = 0;
        source = source + 1 == num_ranks ? 0 : source + 1;
        seg_table.cnt[u] = c;
        seg_table.aux[u] = int(ranges[u] >> 32);
    }
    wave_segments_finish(seg_table);
    DEEPEP_PHASE(1);

    const uint32_t row_bytes = uint32_t(a.hidden) * 2;
    const int num_vec = int(row_bytes / 16);
    const int64_t slots_per_expert = int64_t(max_tokens) * num_ranks;
    const int waves_total = num_blocks * waves;
    const int parts = 1 << a.parts_log2;
    const int num_items = seg_table.total << a.parts_log2;

    for (int item = block * waves + w; item < num_items; item += waves_total) {
        const int row = item >> a.parts_log2, part = item & (parts - 1);
        int seg_first, b;
        const int seg = wave_segments_find(seg_table, row, seg_first, b);
        const int j = row - seg_first;
        const int le = a.expert_of(seg);
        const int s = seg - le * num_ranks;
        if (b < 0 || int64_t(b) + j >= slots_per_expert) continue;  // malformed range: never read past the expert
        const uint8_t* src = a.x + uint64_t(uint32_t(le * slots_per_expert) + uint32_t(b + j)) * row_bytes;
        uint8_t* dst;
        if (s == a.rank)
            dst = a.combine_staging + uint64_t(uint32_t((a.rank * a.num_local_experts + le) * max_tokens + j)) * row_bytes;
        else if (a.combine_send_slots != nullptr)
            dst = a.combine_send_slots + uint64_t(uint32_t(seg * max_tokens + j)) * row_bytes;
        else
            continue;
        int v_begin, v_end;
        row_part_range(num_vec, a.parts_log2, part, v_begin, v_end);
        RowPart<4, kStreamLoad, kStreamStore> piece;
        piece.load(src, v_begin, v_end, lane);
        piece.store(dst, v_begin, lane);
    }
    DEEPEP_PHASE(2);
}

template <bool kStreamLoad, bool kStreamStore>
__device__ __forceinline__ void combine_send_rows(const CombineSendArgs& a, int block, int num_blocks, bool skip_own) {
    if (a.num_local_experts * a.num_ranks <= 4 * kWave)
        combine_send_rows_impl<4, kStreamLoad, kStreamStore>(a, block, num_blocks, skip_own);
    else
        combine_send_rows_impl<16, kStreamLoad, kStreamStore>(a, block, num_blocks, skip_own);
}

// skip_own: the rows owed to this rank itself stay where they are (the reduce reads them from x).
__global__ __launch_bounds__(256) void ll_combine_send_kernel(CombineSendArgs a, bool skip_own) {
    combine_send_rows<false, false>(a, blockIdx.x, gridDim.x, skip_own);
}

// ---------------------------------------------------------------------
// Receive side: one wave = one (token, 1 KiB piece of the output row).
// All K source vectors are loaded before the FMA chain so K 16-byte loads
// are in flight per lane; accumulation order is k = 0..K-1, float32 FMA,
// one rounding to bf16 at the end
// (reference: csrc/kernels/coop_combine_recv.cuh:222-260).
// own_begin != null (single-launch combine): the answers of this rank's own
// experts are read from the expert-output tensor own_x at
// [e_l][own_begin[e_l] + slot] instead of the staging area.
// ---------------------------------------------------------------------
struct CombineRecvArgs {
    const uint8_t* combine_staging;
    const int64_t* topk_idx;
    const float* topk_weights;
    const int32_t* pair_slot;
    int num_tokens, hidden, num_topk, num_experts, max_tokens, pieces_per_row;
    int accumulate;  // non-zero: the sum starts from what `out` already holds
    uint8_t* out;
    // Flat form (rows returned through an all-to-all): combine_staging is one buffer with a row per row
    // sent, in send order; pair (t, k) is answered by row flat_prefix[expert] + slot, or, when the rows of
    // every answering rank start at a slot of flat_slot_rows rows, by row rank * flat_slot_rows + (that
    // minus the first row sent to the rank).  Null flat_prefix: the per-expert staging area.
    const int32_t* flat_prefix;  // [E + 1]
    int64_t flat_rows, flat_slot_rows;
    int experts_per_rank;
};

// What lane k of a wave knows about selection k of its token once the index loads are back.
struct CombineSelection {
    int slot;
    int64_t expert;
    float weight;
};

// Issues the loads of selection `lane`'s (slot, expert, weight): one round of loads for the whole token.
// Nothing here waits for them, so a caller can put other latency (the own-range lookup of the
// single-launch combine) behind the same round trip.
__device__ __forceinline__ CombineSelection combine_load_selection(const CombineRecvArgs& a, uint32_t t) {
    CombineSelection s = {-1, -1, 0.0f};
    const int lane = lane_id();
    if (t < uint32_t(a.num_tokens) && lane < a.num_topk) {
        const int64_t idx = int64_t(t) * a.num_topk + lane;
        s.slot = a.pair_slot[idx];
        s.expert = a.topk_idx[idx];
        s.weight = a.topk_weights[idx];
    }
    return s;
}

template <bool kStream, bool kInTurn>
__device__ __forceinline__ void combine_recv_piece(const CombineRecvArgs& a, uint32_t t, uint32_t piece,
                                                   const CombineSelection& sel, const uint8_t* own_x,
                                                   const int32_t* own_begin, int own_first_expert,
                                                   int num_local_experts, int64_t slots_per_expert) {
    const int lane = lane_id();
    if (t >= uint32_t(a.num_tokens)) return;
    const int64_t row_bytes = int64_t(a.hidden) * 2;
    const int off = int(piece) * 1024 + lane * 16;  // lanes past the row's end read zeros and store nothing
    const int num_topk = a.num_topk;
    const auto out = row_buffer(a.out + int64_t(t) * row_bytes, int(row_bytes));

    DEEPEP_PHASE(0);
    // Lane k works out where selection k's row is; the loop below reads the results back lane by
    // lane, as wave-uniform values.
    uint64_t my_row = 0;
    const float my_weight = sel.weight;
    bool my_live = false;
    if (lane < num_topk) {
        const int slot = sel.slot;
        const int64_t e = sel.expert;
        if (a.flat_prefix != nullptr) {
            // csrc/kernels/efa_kernels.cu:1449-1466: the row's index in send order, flat or inside its rank's slot
            if (slot >= 0 && e >= 0 && e < a.num_experts) {
                const int first = a.flat_prefix[e], next = a.flat_prefix[e + 1];
                int64_t idx = int64_t(first) + slot;
                my_live = first >= 0 && slot < next - first;
                if (a.flat_slot_rows > 0) {
                    const int64_t r = e / a.experts_per_rank;
                    const int64_t within = idx - a.flat_prefix[r * a.experts_per_rank];
                    my_live = my_live && within >= 0 && within < a.flat_slot_rows;
                    idx = r * a.flat_slot_rows + within;
                }
                my_live = my_live && idx < a.flat_rows;
                my_row = reinterpret_cast<uint64_t>(a.combine_staging + idx * row_bytes);
            }
        } else if (slot >= 0 && slot < a.max_tokens && e >= 0 && e < a.num_experts) {
            const uint8_t* row = a.combine_staging + (e * a.max_tokens + slot) * row_bytes;
            my_live = true;
            const int64_t le = e - own_first_expert;
            if (own_begin != nullptr && le >= 0 && le < num_local_experts) {
                const int64_t pos = int64_t(own_begin[le]) + slot;
                my_live = own_begin[le] >= 0 && pos < slots_per_expert;
                row = own_x + (le * slots_per_expert + pos) * row_bytes;
            }
            my_row = reinterpret_cast<uint64_t>(row);
        }
    }
    const uint64_t live_mask = __ballot(my_live);

    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    if (a.accumulate != 0) {  // reference: csrc/kernels/coop_combine_recv.cuh:174-179
        const u32x4 prev = load_row_u32x4<false>(out, off);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[2 * i] = bf16_lo(prev[i]), acc[2 * i + 1] = bf16_hi(prev[i]);
    }

    DEEPEP_PHASE(1);
    add_rows<kStream, true, kInTurn>(my_row, my_weight, live_mask, off, int(row_bytes), acc);
    DEEPEP_PHASE(2);
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = pack_bf16x2(acc[2 * i], acc[2 * i + 1]);
    store_row_u32x4<kStream>(out, off, o);
    DEEPEP_PHASE(3);
}

// kStream: the gathered rows exceed what the caches hold, so they are read (and the result written)
// with the non-temporal hint.  own_x != null: the answers of this rank's own experts are read from
// the expert-output tensor directly (layout_range says where each own segment begins).
// index_blocks > 0: that many workgroups in front of the reduce's build the index of the row return that follows
// (a launch of its own took 3 to 5 us of a large combine).
// Streaming, a workgroup is one wave: nothing holds a wave's slot once it is done (4096 tokens, eight rows of 14336
// bytes each, 90.5 -> 88.7 us, 6.0 TB/s; two to fourteen waves 91 to 95, neighbouring tokens on one XCD no gain).
// Eight waves a SIMD while the rows stay in the caches: 820 to 1000 tokens of 5120 at top-4 4 % less than with six, else the
// same.  Streaming, six serve HBM as well or better (87.5 us against 87.8 at 4096 tokens).
// It streams from 32 MB of rows on, which nobody reads again.  A whole exchange to 8 ranks on three sets of buffers in turn,
// from 192 MB on / from 32: 700 tokens of 7168 93.6 / 90.5 us, 1000 of 4096 81.6 / 78.8, 1500 of 5120 at top-6 113.4 / 109.8,
// 2047 of 4096 133.8 / 131.2, 400 of 7168 (44 MB) 55 from 48 MB on and 51.4 so; 256 of 7168 (28 MB) 38.6 / 39.5 with it.  Behind a
// read of 512 MB the reduce alone 12.0 / 11.7 at 400 tokens and 19.1 / 19.0 at 700, behind a write 20.1 / 11.5 and 34.2 / 19.3.
constexpr int64_t kReduceStreamBytes = int64_t(32) << 20;
template <bool kStream>
__global__ __launch_bounds__(256) void ll_combine_recv_kernel(CombineRecvArgs a, const uint8_t* own_x,
                                                              const int64_t* layout_range, int rank,
                                                              int num_local_experts, int num_ranks, uint32_t waves,
                                                              CombineIndexArgs index, int index_blocks) {
    extern __shared__ int32_t own_begin[];  // [E_l], with own_x only; index workgroups: [segments + 1]
    __shared__ int32_t index_wave_totals[kMaxBlockWaves];
    if (int(blockIdx.x) < index_blocks) {
        combine_index_block(index, blockIdx.x, own_begin, index_wave_totals);
        return;
    }
    const uint32_t item = (blockIdx.x - index_blocks) * waves + wave_in_block(), pieces = a.pieces_per_row;
    const uint32_t t = item / pieces, piece = item - t * pieces;
    const CombineSelection sel = combine_load_selection(a, t);  // in flight while the own ranges are fetched
    if (own_x != nullptr) {
        for (int le = threadIdx.x; le < num_local_experts; le += int(waves) * kWave) {
            const int64_t lr = layout_range[le * num_ranks + rank];
            own_begin[le] = (lr & 0xffffffffll) > 0 ? int(lr >> 32) : 0;
        }
        lds_barrier();
    }
    combine_recv_piece<kStream, !kStream>(a, t, piece, sel, own_x, own_x != nullptr ? own_begin : nullptr,
                                          rank * num_local_experts, num_local_experts, int64_t(a.max_tokens) * num_ranks);
}

__global__ __launch_bounds__(256) void ll_combine_index_kernel(CombineIndexArgs index) {
    extern __shared__ int32_t flat[];  // [segments + 1]
    __shared__ int32_t wave_totals[kMaxBlockWaves];
    combine_index_block(index, blockIdx.x, flat, wave_totals);
}

// ---------------------------------------------------------------------
// Single-launch combine (combine_in_one_launch() says for which batches): the reduce workgroups
// and the row-return workgroups of the two kernels above in one grid.  No
// workgroup waits on another: the reduce reads the answers of this rank's own
// experts straight from x (layout_range says where each segment begins), so the
// row return only has to move the rows owed to other ranks.
// (The reference's combine is one kernel with a send and a receive phase as
// well: csrc/kernels/coop_combine_send.cuh:37, coop_combine_recv.cuh:72.)
// kInTurn: eight waves a SIMD, for grids that the chip then holds at once.  128 tokens are 1616 to 1646 workgroups: with
// six the last row returns start 4.9 us into a kernel of 5.9 (7.7 of 8.7 after a flush), with eight 1.7 (1.5).  A step of
// 128 tokens takes the same, of 280 x 5120 at top-4 14.7 -> 14.0 us, 200 x 5120 at top-6 17.5 -> 16.4, 280 x 4096 21.2 -> 20.6,
// 160 x 7168 to 32 ranks 20.7 -> 20.1.  Beyond one round it depends on how full the last one is: 1.1 to 1.5 rounds of eight
// gain 2 to 4 %, 1.7 to 2.05 lose as much (577 x 5120 at top-4 29.1 -> 30.2), more than three lose 0 to 1 %: six there.
// ---------------------------------------------------------------------
constexpr int64_t kWorkgroupsAtOnce = 256 * 8;  // compute units, workgroups of four waves on each
// Which accesses of the single-launch combine stream.  Past 48 MB of traffic its stores and the gathered rows, which
// nobody touches again, while the rows to be returned, which the experts have just written, are read the ordinary way;
// past 192 MB, where nothing survives from one kernel to the next, those too.  The hint keeps the combine from displacing
// what its neighbours left, and from waiting for their dirty lines to be written back.  Microseconds of dispatch + combine
// without it below 192 MB / with it, behind steps on other buffers (three in turn; the wider one, called from C++), and of
// their kernels behind a read (R) and behind a write (W) of 512 MB each:
//   150 x 7168 to 32 ranks     24.8 / 24.2    R 20.4 / 20.2    W 28.8 / 24.9
//   256 x 4096                 25.1 / 23.1    R 20.2 / 19.4    W 26.9 / 22.4
//   300 x 7168                 46.6 / 38.4    R 34.9 / 34.4    W 51.2 / 40.6
//   500 x 2048                 26.6 / 24.0    R 21.5 / 20.9    W 28.4 / 24.1
//   700 x 4096                 54.6 / 45.1    R 43.6 / 44.6    W 63.7 / 51.9    (the dispatch's own share: common.hpp)
//   900 x 2048                 42.5 / 38.8    R 33.5 / 33.0    W 47.0 / 38.6
// Replayed on one set of buffers, all of it still cached, it costs 150 to 180 tokens 5 to 7 % and gains from 700 on.
// Below, 128 x 7168 (46 MB) gains 3 % on other buffers and loses 2 % behind a read, 256 x 5120 at top-4 (33 MB) and 77 x 5120
// lose 2 % both ways.  The hint on the rows to be returned as well: 128 and 150 tokens 3 % slower than without any, 256 x
// 4096 24.3 us, 500 x 2048 25.8, 700 x 4096 45.7, but 300 x 7168 37.2 and behind a write another 8 to 13 % less.
constexpr int64_t kGatherStreamBytes = int64_t(48) << 20;
// Without a row return the gathered rows are all there is, and the line lies at 18 MB of them.  Steps in microseconds without
// the hint / with it, on three sets of buffers in turn and on one, and the combine alone behind a write of 512 MB (behind a read
// the two differ by no more than two runs of one):
//   128 x 7168 (15 MB)  15.7 / 16.4   15.1 / 15.4   14.5 /  8.9     256 x 7168 (29 MB)  23.7 / 22.9   21.1 / 22.6   18.9 / 11.2
//   500 x 2048 (16 MB)  18.1 / 18.6   17.1 / 17.5   12.7 /  9.0     300 x 7168 (34 MB)  26.8 / 24.8   22.9 / 24.5   21.1 / 12.2
//   150 x 7168 (17 MB)  16.8 / 17.7   16.0 / 16.8   14.0 /  9.8     509 x 4096 (33 MB)  28.3 / 24.6   22.4 / 23.2   17.6 / 11.8
//   180 x 7168 (21 MB)  19.7 / 19.1   17.7 / 18.7   15.2 /  9.6     700 x 4096 (46 MB)  31.7 / 29.6   27.8 / 28.8   25.3 / 14.6
constexpr int64_t kGatherAloneStreamBytes = int64_t(18) << 20;

// kStream: stores and gathered rows; kStreamRows: the rows to be returned as well.
template <bool kStream, bool kStreamRows, bool kInTurn>
__device__ __forceinline__ void combine_fused_block(const CombineSendArgs& sa, const CombineRecvArgs& ra,
                                                    int num_recv_blocks, int32_t* dyn_lds) {
    // dyn_lds: reduce workgroups, own_begin[E_l]
    const int block = blockIdx.x;
    if (block < num_recv_blocks) {
        // the token's index loads and the own-range loads go out together: one memory round trip
        // before the row loads instead of two
        const uint32_t item = uint32_t(block) * 4 + wave_in_block(), pieces = ra.pieces_per_row;
        const uint32_t t = item / pieces, piece = item - t * pieces;
        const CombineSelection sel = combine_load_selection(ra, t);
        for (int le = threadIdx.x; le < sa.num_local_experts; le += 256) {
            const int64_t lr = sa.layout_range[le * sa.num_ranks + sa.rank];
            dyn_lds[le] = (lr & 0xffffffffll) > 0 ? int(lr >> 32) : 0;
        }
        lds_barrier();
        combine_recv_piece<kStream, kInTurn>(ra, t, piece, sel, sa.x, dyn_lds, sa.rank * sa.num_local_experts,
                                             sa.num_local_experts, int64_t(sa.max_tokens) * sa.num_ranks);
    } else {
        combine_send_rows<kStreamRows, kStream>(sa, block - num_recv_blocks, int(gridDim.x) - num_recv_blocks, true);
    }
}

template <bool kStream, bool kInTurn>
__global__ __launch_bounds__(256) void ll_combine_fused_kernel(CombineSendArgs sa, CombineRecvArgs ra,
                                                               int num_recv_blocks) {
    extern __shared__ int32_t dyn_lds[];
    combine_fused_block<kStream, false, kInTurn>(sa, ra, num_recv_blocks, dyn_lds);
}

__global__ __launch_bounds__(256) void ll_combine_fused_past_caches_kernel(CombineSendArgs sa, CombineRecvArgs ra,
                                                                           int num_recv_blocks) {
    extern __shared__ int32_t dyn_lds[];
    combine_fused_block<true, true, false>(sa, ra, num_recv_blocks, dyn_lds);
}

// ---------------------------------------------------------------------
// Send side for an all-to-all shaped transport: the live expert-output rows in
// arrival order, which is contiguous per destination rank.  Record i of the
// exchange metadata names the row (padded_index[i] picks the record whose packed
// row is read, record_packed_row says where the receive side put it) and its place
// in the flat buffer (combine_send_offset[i]); reference:
// send_buffer[combine_send_offset[i]] = expert_x[padded_index[i]]
// (csrc/kernels/coop_combine_send.cuh:37-170; torch form deep_ep/buffer.py:2601-2608).
// With a table of peer buffers the row skips the send buffer and goes straight to
// its place in the destination's receive buffer, behind what that rank sent to the
// ranks below this one (combine_remote_recv_offset,
// csrc/transport/ll_pipeline.cpp:1283-1295; the reference's peer stores:
// coop_combine_send.cuh:205-246).  One workgroup per record, walked like the rows of ll_rows_flat_kernel: HBM
// bounds it, and neighbouring records are neighbouring rows on both sides.  Up to 512 threads: with twice the trips in
// front of a row that a described one has, 896 for a row of 14336 bytes are the slower form behind an ordered receive
// (16376 rows 77 us against 75.4, 1024 rows 6.9 against 6.4), until the rows are so many that a vector a thread pays as it
// does there: 40000 rows 176 us with up to 512 threads and 171.6 with 896, 160000 746 and 693 (two vectors a thread 755),
// 320000 1537 and 1399.
// 16376 rows of 14336 bytes 78.7 -> 75.4 us (6.2 TB/s), 1024 rows 7.7 -> 6.4, against two vectors a thread and the
// record behind the number of records.
// From 24 MB on (both directions) its stores stream, from 48 MB the loads too.  A whole exchange on three sets of buffers
// in turn, from 192 MB on / so, other lines alike: 128 tokens of 7168 to 8 ranks 26.6 / 24.9 us, 256 of 4096 to 32 30.5 / 29.1,
// 256 of 7168 to 16 46.4 / 39.5, 400 to 8 62.4 / 59.0, 1500 of 5120 at top-6 113.4 / 109.4; stores alone also past 48 MB 42.4 for
// the 256, 60.8 for the 400 and 87.7 instead of 81 for 700.  Alone behind a read of 512 MB 256 tokens 13.3 / 12.9, 400 18.5 /
// 18.6, 128 7.4 / 7.6, behind a write 18.1 / 13.4, 27.9 / 19.1, 9.4 / 9.9; an exchange of 256 on one set of buffers 35.5 / 38.4.
// ---------------------------------------------------------------------
constexpr int64_t kReturnStreamBytes = int64_t(48) << 20, kReturnStreamStoreBytes = int64_t(24) << 20;

struct CombineByDestPeers {  // direct delivery
    uint8_t* const* peer_recv;   // [R] device pointers, or null
    const int64_t* peer_rows;    // [R] rows each peer buffer holds
    const int32_t* recv_counts;
    const int64_t* remote_offset;
    const uint32_t* source_rank;
    int num_ranks;
};

template <bool kStreamLoad, bool kStreamStore, bool kPeers>
__global__ __launch_bounds__(1024) void ll_combine_send_by_dest_kernel(
    const uint32_t* __restrict__ num_recv_tokens, const uint32_t* __restrict__ padded_index,
    const int32_t* __restrict__ record_packed_row, const uint32_t* __restrict__ combine_send_offset,
    uint32_t row_capacity, uint32_t x_rows, const uint8_t* __restrict__ x, uint8_t* __restrict__ send_flat, int num_vec,
    int threads, uint32_t grid, CombineByDestPeers peers) {
    const uint64_t row_bytes = uint64_t(num_vec) * 16;
    uint32_t block = blockIdx.x, i = flat_row_of_block(block);
    // The record is fetched together with the number of records (both sides of the bound are memory the
    // tables have), and padded_index[i] is i whenever the records come from deepep_ll_exchange_metadata, so
    // the packed row is fetched for that guess as well and again only if the guess was wrong: one round trip
    // in front of the row loads instead of three.
    const uint32_t at = i < row_capacity ? i : row_capacity - 1;
    uint32_t records = num_recv_tokens[1], p = padded_index[at], src_row = uint32_t(record_packed_row[at]);
    uint32_t offset = combine_send_offset[at];
    await_scalars(records, p, src_row, offset);
    if (records > row_capacity) records = row_capacity;
    for (;;) {
        if (i < records && p < row_capacity) {
            if (p != i) src_row = uint32_t(record_packed_row[p]);
            uint8_t* dst = nullptr;
            if constexpr (!kPeers) {
                if (offset < row_capacity) dst = send_flat + offset * row_bytes;
            } else {
                const uint32_t s = peers.source_rank[i];
                if (s < uint32_t(peers.num_ranks)) {
                    // the record's place among the rows of its source: offset minus the rows of the lower sources
                    const int lane = lane_id();
                    int part = 0;
                    for (int r = lane; r < int(s); r += kWave) part += peers.recv_counts[r] < 0 ? 0 : peers.recv_counts[r];
                    const int64_t j = int64_t(offset) - __builtin_amdgcn_readlane(wave_inclusive_sum(part), kWave - 1);
                    const int64_t at_peer = peers.remote_offset[s] + j;
                    if (j >= 0 && j < peers.recv_counts[s] && at_peer >= 0 && at_peer < peers.peer_rows[s])
                        dst = peers.peer_recv[s] + at_peer * row_bytes;
                }
            }
            if (dst != nullptr && src_row < x_rows)  // < 0: the record has no row
                block_copy_row<1, kStreamLoad, kStreamStore>(x + src_row * row_bytes, dst, num_vec, threadIdx.x, threads);
        }
        if (uint64_t(block) + grid >= flat_rounds_end(records)) break;
        block += grid, i = flat_row_of_block(block);
        if (i < records) p = padded_index[i], src_row = uint32_t(record_packed_row[i]), offset = combine_send_offset[i];
    }
}

static CombineSendArgs make_combine_send_args(const void* x, const int64_t* layout_range, int hidden, int num_experts,
                                              int num_ranks, int rank, int max_tokens, void* combine_staging,
                                              void* combine_send_slots, int64_t expected_rows) {
    CombineSendArgs sa;
    sa.x = reinterpret_cast<const uint8_t*>(x);
    sa.layout_range = layout_range;
    sa.hidden = hidden, sa.num_local_experts = num_experts / num_ranks, sa.num_ranks = num_ranks, sa.rank = rank;
    sa.expert_of = make_rank_divider(num_ranks);
    sa.max_tokens = max_tokens;
    sa.parts_log2 = choose_row_parts_log2(estimated_rows(expected_rows, num_experts, max_tokens), int64_t(hidden) * 2,
                                          num_experts);
    sa.combine_staging = reinterpret_cast<uint8_t*>(combine_staging);
    sa.combine_send_slots = reinterpret_cast<uint8_t*>(combine_send_slots);
    return sa;
}

static CombineRecvArgs make_combine_recv_args(const void* combine_staging, const int64_t* topk_idx,
                                              const float* topk_weights, const int32_t* pair_slot, int num_tokens,
                                              int hidden, int num_topk, int num_experts, int max_tokens, int accumulate,
                                              void* out) {
    CombineRecvArgs ra;
    ra.combine_staging = reinterpret_cast<const uint8_t*>(combine_staging);
    ra.topk_idx = topk_idx, ra.topk_weights = topk_weights, ra.pair_slot = pair_slot;
    ra.num_tokens = num_tokens, ra.hidden = hidden, ra.num_topk = num_topk, ra.num_experts = num_experts;
    ra.max_tokens = max_tokens, ra.pieces_per_row = (hidden * 2 + 1023) / 1024;
    ra.accumulate = accumulate;
    ra.out = reinterpret_cast<uint8_t*>(out);
    ra.flat_prefix = nullptr, ra.flat_rows = 0, ra.flat_slot_rows = 0, ra.experts_per_rank = 1;
    return ra;
}

static int check_combine_send_args(const void* x, const int64_t* layout_range, int hidden, int num_experts,
                                   int num_ranks, int rank, int max_tokens, const void* combine_staging,
                                   const void* combine_send_slots) {
    EP_HOST_ASSERT(hidden > 0 && hidden % 128 == 0);
    EP_HOST_ASSERT(num_ranks > 0 && num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(rank >= 0 && rank < num_ranks);
    EP_HOST_ASSERT(max_tokens > 0);
    EP_HOST_ASSERT(num_experts <= 1024);
    EP_HOST_ASSERT(x != nullptr && layout_range != nullptr && combine_staging != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(layout_range) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(combine_staging) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(combine_send_slots) & 15) == 0);
    EP_HOST_ASSERT(int64_t(num_experts) * max_tokens < (int64_t(1) << 31));
    return 0;
}

static int check_combine_recv_args(const void* combine_staging, const int64_t* topk_idx, const float* topk_weights,
                                   const int32_t* pair_slot, int num_tokens, int hidden, int num_topk,
                                   int num_experts, int max_tokens, const void* out) {
    EP_HOST_ASSERT(num_tokens >= 0 && hidden > 0 && hidden % 128 == 0 && num_topk > 0);
    EP_HOST_ASSERT(num_experts > 0 && max_tokens > 0);
    if (num_tokens == 0) return 0;
    EP_HOST_ASSERT(combine_staging != nullptr && topk_idx != nullptr && topk_weights != nullptr &&
                   pair_slot != nullptr && out != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(combine_staging) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(out) & 15) == 0);
    EP_HOST_ASSERT(int64_t(num_tokens) * ((hidden * 2 + 1023) / 1024) < (int64_t(1) << 31));
    return 0;
}

}  // namespace deepep

using namespace deepep;

extern "C" {

// The index and the flat copy of a large row return, in `workspace`.
static int make_combine_index(const int64_t* layout_range, int num_experts, int num_ranks, int rank,
                              int num_max_dispatch_tokens_per_rank, bool skip_own, void* workspace,
                              size_t workspace_bytes, CombineIndexArgs& index) {
    EP_HOST_ASSERT(workspace_bytes >= size_t(segment_workspace_bytes(num_experts, num_max_dispatch_tokens_per_rank)));
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(workspace) & 15) == 0);
    index.layout_range = layout_range;
    index.num_local_experts = num_experts / num_ranks, index.num_ranks = num_ranks, index.rank = rank;
    index.max_tokens = num_max_dispatch_tokens_per_rank, index.skip_own = skip_own;
    index.flat_out = reinterpret_cast<int32_t*>(workspace);
    index.desc = reinterpret_cast<RowDesc*>(reinterpret_cast<uint8_t*>(workspace) +
                                            (((int64_t(num_experts) + 1) * 4 + 255) & ~int64_t(255)));
    return 0;
}

static int launch_combine_rows(const CombineIndexArgs& index, const void* x, int hidden, void* combine_staging,
                               void* combine_send_slots, int64_t expected_rows, hipStream_t hs) {
    const int num_experts = index.num_local_experts * index.num_ranks, num_vec = hidden * 2 / 16;
    const int64_t max_rows = int64_t(num_experts) * index.max_tokens;
    const int64_t rows = estimated_rows(expected_rows, num_experts, index.max_tokens);
    launch_rows_flat(index.flat_out + num_experts, index.desc, max_rows,
                     index.skip_own ? rows - rows / index.num_ranks : rows, x, int64_t(hidden) * 2, num_vec,
                     combine_send_slots, combine_staging, int64_t(hidden) * 2, nullptr, hs);
    EP_LAUNCH_CHECK();
    return 0;
}

// skip_own: the rows owed to this rank itself are not moved (the reduce will read them from x).
static int launch_combine_send(const void* x, const int64_t* layout_range, int hidden, int num_experts, int num_ranks,
                               int rank, int num_max_dispatch_tokens_per_rank, void* combine_staging,
                               void* combine_send_slots, int64_t expected_rows, void* workspace,
                               size_t workspace_bytes, bool skip_own, void* stream) {
    if (int rc = check_combine_send_args(x, layout_range, hidden, num_experts, num_ranks, rank,
                                         num_max_dispatch_tokens_per_rank, combine_staging, combine_send_slots))
        return rc;
    const int64_t max_rows = int64_t(num_experts) * num_max_dispatch_tokens_per_rank;
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    const bool large = estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank) > kLargeBatchRows;
    if (large && workspace != nullptr) {
        CombineIndexArgs index;
        if (int rc = make_combine_index(layout_range, num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank,
                                        skip_own, workspace, workspace_bytes, index))
            return rc;
        launch(ll_combine_index_kernel, num_experts, 256, size_t(num_experts + 1) * sizeof(int32_t), hs, index);
        EP_LAUNCH_CHECK();
        return launch_combine_rows(index, x, hidden, combine_staging, combine_send_slots, expected_rows, hs);
    }
    const CombineSendArgs sa = make_combine_send_args(x, layout_range, hidden, num_experts, num_ranks, rank,
                                                      num_max_dispatch_tokens_per_rank, combine_staging,
                                                      combine_send_slots, expected_rows);
    int64_t blocks = ((max_rows << sa.parts_log2) + 3) / 4;
    const int64_t cap = large ? 4096 : 1024;
    if (blocks > cap) blocks = cap;
    launch(ll_combine_send_kernel, dim3(unsigned(blocks)), 256, 0, hs, sa, skip_own);
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_ll_combine_send(const void* x, const int64_t* layout_range, int hidden, int num_experts, int num_ranks,
                           int rank, int num_max_dispatch_tokens_per_rank, void* combine_staging,
                           void* combine_send_slots, int64_t expected_rows, void* workspace, size_t workspace_bytes,
                           void* stream) {
    clear_error();
    return launch_combine_send(x, layout_range, hidden, num_experts, num_ranks, rank,
                               num_max_dispatch_tokens_per_rank, combine_staging, combine_send_slots, expected_rows,
                               workspace, workspace_bytes, false, stream);
}

static void launch_reduce(const CombineRecvArgs& ra, const uint8_t* own, const int64_t* layout_range, int rank,
                          int num_local_experts, int num_ranks, const CombineIndexArgs* index, hipStream_t hs) {
    const bool stream_rows = int64_t(ra.num_tokens) * ra.num_topk * ra.hidden * 2 > kReduceStreamBytes;
    const int waves = stream_rows ? 1 : 4;
    const int index_blocks = index != nullptr ? index->num_local_experts * index->num_ranks : 0;
    const CombineIndexArgs ia = index != nullptr ? *index : CombineIndexArgs{};
    const int64_t blocks = index_blocks + (int64_t(ra.num_tokens) * ra.pieces_per_row + waves - 1) / waves;
    const size_t lds = size_t(index_blocks > 0 ? index_blocks + 1 : num_local_experts) * sizeof(int32_t);
    if (stream_rows)
        launch(ll_combine_recv_kernel<true>, dim3(unsigned(blocks)), waves * kWave, lds, hs,
            ra, own, layout_range, rank, num_local_experts, num_ranks, uint32_t(waves), ia, index_blocks);
    else
        launch(ll_combine_recv_kernel<false>, dim3(unsigned(blocks)), waves * kWave, lds, hs,
            ra, own, layout_range, rank, num_local_experts, num_ranks, uint32_t(waves), ia, index_blocks);
}

// own_x != null: the answers of this rank's own experts are read from own_x at the positions
// layout_range gives, instead of from combine_staging.
static int launch_combine_recv(const void* combine_staging, const int64_t* topk_idx, const float* topk_weights,
                               const int32_t* pair_slot, int num_tokens, int hidden, int num_topk, int num_experts,
                               int num_max_dispatch_tokens_per_rank, int accumulate, void* out, const void* own_x,
                               const int64_t* layout_range, int rank, int num_ranks, const CombineIndexArgs* index,
                               void* stream) {
    if (int rc = check_combine_recv_args(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens, hidden,
                                         num_topk, num_experts, num_max_dispatch_tokens_per_rank, out))
        return rc;
    if (num_tokens == 0) return 0;
    const CombineRecvArgs ra = make_combine_recv_args(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens,
                                                      hidden, num_topk, num_experts,
                                                      num_max_dispatch_tokens_per_rank, accumulate, out);
    launch_reduce(ra, reinterpret_cast<const uint8_t*>(own_x), layout_range, rank,
                  own_x != nullptr ? num_experts / num_ranks : 0, num_ranks, index,
                  reinterpret_cast<hipStream_t>(stream));
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_ll_combine_recv(const void* combine_staging, const int64_t* topk_idx, const float* topk_weights,
                           const int32_t* pair_slot, int num_tokens, int hidden, int num_topk, int num_experts,
                           int num_max_dispatch_tokens_per_rank, int accumulate, void* out, void* stream) {
    clear_error();
    return launch_combine_recv(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens, hidden, num_topk,
                               num_experts, num_max_dispatch_tokens_per_rank, accumulate, out, nullptr, nullptr, 0, 1,
                               nullptr, stream);
}

int deepep_ll_combine_send_by_dest(const void* x, const int32_t* record_packed_row, const uint32_t* source_rank,
                                   const uint32_t* padded_index, const uint32_t* combine_send_offset,
                                   const uint32_t* num_recv_tokens, int64_t row_capacity, int hidden, int num_experts,
                                   int num_ranks, int num_max_dispatch_tokens_per_rank, void* send_flat,
                                   const int32_t* recv_counts, const int64_t* combine_remote_recv_offset,
                                   void* const* peer_recv_flat, const int64_t* peer_recv_rows,
                                   int64_t expected_rows, void* stream) {
    clear_error();
    EP_HOST_ASSERT(hidden > 0 && hidden % 128 == 0);
    EP_HOST_ASSERT(num_ranks > 0 && num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(num_max_dispatch_tokens_per_rank > 0);
    EP_HOST_ASSERT(row_capacity >= 0 && row_capacity < (int64_t(1) << 31));
    if (row_capacity == 0) return 0;
    EP_HOST_ASSERT(x != nullptr && record_packed_row != nullptr && padded_index != nullptr &&
                   combine_send_offset != nullptr && num_recv_tokens != nullptr);
    const bool direct = peer_recv_flat != nullptr;
    EP_HOST_ASSERT(direct || send_flat != nullptr);
    EP_HOST_ASSERT(!direct || (source_rank != nullptr && recv_counts != nullptr &&
                               combine_remote_recv_offset != nullptr && peer_recv_rows != nullptr));
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(send_flat) & 15) == 0);
    CombineByDestPeers peers;
    peers.peer_recv = reinterpret_cast<uint8_t* const*>(peer_recv_flat), peers.peer_rows = peer_recv_rows;
    peers.recv_counts = recv_counts, peers.remote_offset = combine_remote_recv_offset;
    peers.source_rank = source_rank, peers.num_ranks = num_ranks;
    // grid from the rows expected, not from the capacity (an idle workgroup is not free)
    const int64_t rows = expected_rows > 0 && expected_rows < row_capacity ? expected_rows : row_capacity;
    const int64_t sized_for = flat_rows_expected(expected_rows, row_capacity);
    const int num_vec = hidden * 2 / 16, threads = flat_row_threads(num_vec, sized_for > 32768 ? 1024 : 512);
    const unsigned grid = flat_grid_blocks(sized_for, row_capacity, threads);
    const int64_t x_rows = std::min(int64_t(num_experts) * num_max_dispatch_tokens_per_rank, int64_t(1) << 31);
#define DEEPEP_LAUNCH_BY_DEST(LOAD, STORE, PEERS)                                                                       \
    launch(ll_combine_send_by_dest_kernel<LOAD, STORE, PEERS>, grid, threads, 0, reinterpret_cast<hipStream_t>(stream),     \
        num_recv_tokens, padded_index, record_packed_row, combine_send_offset, uint32_t(row_capacity),                  \
        uint32_t(x_rows), reinterpret_cast<const uint8_t*>(x),                                                          \
        reinterpret_cast<uint8_t*>(send_flat), num_vec, threads, grid, peers)
    const int64_t traffic = 2 * rows * hidden * 2;
    if (traffic > kReturnStreamBytes) {
        if (peer_recv_flat != nullptr) DEEPEP_LAUNCH_BY_DEST(true, true, true);
        else DEEPEP_LAUNCH_BY_DEST(true, true, false);
    } else if (traffic > kReturnStreamStoreBytes) {
        if (peer_recv_flat != nullptr) DEEPEP_LAUNCH_BY_DEST(false, true, true);
        else DEEPEP_LAUNCH_BY_DEST(false, true, false);
    } else {
        if (peer_recv_flat != nullptr) DEEPEP_LAUNCH_BY_DEST(false, false, true);
        else DEEPEP_LAUNCH_BY_DEST(false, false, false);
    }
#undef DEEPEP_LAUNCH_BY_DEST
    EP_LAUNCH_CHECK();
    return 0;
}

int deepep_ll_combine_recv_flat(const void* recv_flat, int64_t recv_flat_rows, int64_t slot_rows,
                                const int32_t* send_expert_prefix, const int64_t* topk_idx,
                                const float* topk_weights, const int32_t* pair_slot, int num_tokens, int hidden,
                                int num_topk, int num_experts, int num_ranks, int num_max_dispatch_tokens_per_rank,
                                int accumulate, void* out, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_ranks > 0 && num_experts > 0 && num_experts % num_ranks == 0);
    EP_HOST_ASSERT(recv_flat_rows >= 0 && slot_rows >= 0);
    EP_HOST_ASSERT(slot_rows == 0 || slot_rows * num_ranks <= recv_flat_rows);
    if (int rc = check_combine_recv_args(recv_flat, topk_idx, topk_weights, pair_slot, num_tokens, hidden, num_topk,
                                         num_experts, num_max_dispatch_tokens_per_rank, out))
        return rc;
    if (num_tokens == 0) return 0;
    EP_HOST_ASSERT(send_expert_prefix != nullptr);
    CombineRecvArgs ra = make_combine_recv_args(recv_flat, topk_idx, topk_weights, pair_slot, num_tokens, hidden,
                                                num_topk, num_experts, num_max_dispatch_tokens_per_rank, accumulate,
                                                out);
    ra.flat_prefix = send_expert_prefix, ra.flat_rows = recv_flat_rows, ra.flat_slot_rows = slot_rows;
    ra.experts_per_rank = num_experts / num_ranks;
    launch_reduce(ra, nullptr, nullptr, 0, 0, 1, nullptr, reinterpret_cast<hipStream_t>(stream));
    EP_LAUNCH_CHECK();
    return 0;
}

// Whether a combine whose rows are to be returned runs as one launch.  Up to kLargeBatchRows rows always.  Beyond, while
// the rows returned and the tokens' rows stay within 132 MB: there the rows are moved beside the reduce's loads and the
// step has one launch less, past it the flat copy's rate is worth more.  Not where far more rows come in than the tokens
// send out (the hottest experts' rank: the reduce is too short to hide anything), nor for many rows of less than 2 KB.
// Microseconds of a dispatch and a combine, one launch against two (rows, row size; 8 ranks x 8 experts unless given):
//    8800 of  4 KB  45.3 /  46.9      8800 of 14 KB (142 MB)   109.4 / 106.7     31786 of 1 KB     59.6 /  57.9
//   14400 of  4 KB  60.8 /  62.4     10400 of 14 KB (16 ranks) 127.3 / 125.5     31786 of 256 B    47.9 /  45.5
//    8800 of  8 KB  70.3 /  71.4     12000 of 14 KB (194 MB)   140.9 / 138.1     10358 of 1 KB     33.5 /  34.5
//   12800 of  8 KB  94.0 /  94.0      9200 of 14 KB (top-4)    114.6 / 114.2
//   16800 of  8 KB 121.8 / 116.6      9000 of 10 KB (top-6)     88.1 /  89.7
//   28000 of  4 KB 101.8 / 101.8     10000 of 10 KB (top-4)     93.6 /  94.6
//   skewed, 64 ranks: 10324 rows for 7200 selections 130.8 / 137.8, 13638 for 1600 130.0 / 119.8
// Past 256 experts, whose rows are not moved in parts (choose_row_parts_log2), up to 220 MB.
static bool combine_in_one_launch(int64_t rows, int num_tokens, int num_topk, int64_t row_bytes, int num_experts) {
    if (rows <= kLargeBatchRows) return true;
    const int64_t most = int64_t(num_experts <= 4 * kWave ? 132 : 220) << 20;
    return rows <= 2 * int64_t(num_tokens) * num_topk && (rows + num_tokens) * row_bytes <= most &&
           (row_bytes >= 2048 || rows <= 12288);
}

int deepep_ll_combine(const void* x, const int64_t* layout_range, const int64_t* topk_idx, const float* topk_weights,
                      const int32_t* pair_slot, int num_tokens, int hidden, int num_topk, int num_experts,
                      int num_ranks, int rank, int num_max_dispatch_tokens_per_rank, int accumulate,
                      void* combine_staging, void* combine_send_slots, void* out, int64_t expected_rows,
                      void* workspace, size_t workspace_bytes, void* stream) {
    clear_error();
    const int64_t max_rows = int64_t(num_experts) * num_max_dispatch_tokens_per_rank;
    const int64_t estimated = estimated_rows(expected_rows, num_experts, num_max_dispatch_tokens_per_rank);
    const bool large = estimated > kLargeBatchRows;
    if (large && (combine_send_slots == nullptr ||
                  !combine_in_one_launch(estimated, num_tokens, num_topk, int64_t(hidden) * 2, num_experts))) {
        // the two phases back to back, with the single launch's shortcut: the rows owed to this rank
        // itself are not moved, the reduce reads them from x.  Without send slots (zero copy: the transport
        // sends layout_range's ranges straight from x) there is nothing to return.
        if (int rc = check_combine_send_args(x, layout_range, hidden, num_experts, num_ranks, rank,
                                             num_max_dispatch_tokens_per_rank, combine_staging, combine_send_slots))
            return rc;
        // The reduce goes first and builds the row return's index on the way, unless there is nothing to reduce
        // or no memory for an index.
        const bool index_in_reduce = combine_send_slots != nullptr && workspace != nullptr && num_tokens > 0;
        CombineIndexArgs index;
        if (index_in_reduce) {
            if (int rc = make_combine_index(layout_range, num_experts, num_ranks, rank,
                                            num_max_dispatch_tokens_per_rank, true, workspace, workspace_bytes, index))
                return rc;
        } else if (combine_send_slots != nullptr) {
            if (int rc = launch_combine_send(x, layout_range, hidden, num_experts, num_ranks, rank,
                                             num_max_dispatch_tokens_per_rank, combine_staging, combine_send_slots,
                                             expected_rows, workspace, workspace_bytes, true, stream))
                return rc;
        }
        if (int rc = launch_combine_recv(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens, hidden,
                                         num_topk, num_experts, num_max_dispatch_tokens_per_rank, accumulate, out, x,
                                         layout_range, rank, num_ranks, index_in_reduce ? &index : nullptr, stream))
            return rc;
        if (!index_in_reduce) return 0;
        return launch_combine_rows(index, x, hidden, combine_staging, combine_send_slots, expected_rows,
                                   reinterpret_cast<hipStream_t>(stream));
    }
    if (int rc = check_combine_send_args(x, layout_range, hidden, num_experts, num_ranks, rank,
                                         num_max_dispatch_tokens_per_rank, combine_staging, combine_send_slots))
        return rc;
    if (int rc = check_combine_recv_args(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens, hidden,
                                         num_topk, num_experts, num_max_dispatch_tokens_per_rank, out))
        return rc;
    if (large && workspace != nullptr) {  // not needed in one launch: held to the same rules
        CombineIndexArgs index;
        if (int rc = make_combine_index(layout_range, num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank,
                                        true, workspace, workspace_bytes, index))
            return rc;
    }
    const CombineSendArgs sa = make_combine_send_args(x, layout_range, hidden, num_experts, num_ranks, rank,
                                                      num_max_dispatch_tokens_per_rank, combine_staging,
                                                      combine_send_slots, expected_rows);
    const CombineRecvArgs ra = make_combine_recv_args(combine_staging, topk_idx, topk_weights, pair_slot, num_tokens,
                                                      hidden, num_topk, num_experts,
                                                      num_max_dispatch_tokens_per_rank, accumulate, out);
    const int64_t recv_blocks = (int64_t(num_tokens) * ra.pieces_per_row + 3) / 4;
    int64_t rows = expected_rows > 0 ? expected_rows : int64_t(num_max_dispatch_tokens_per_rank) * num_topk;
    rows += rows / 8 + 16;
    if (rows > max_rows) rows = max_rows;
    int64_t send_blocks = combine_send_slots != nullptr ? ((rows << sa.parts_log2) + 3) / 4 : 0;
    // A wave for each row part: one that goes round finds its next row behind two trips to memory.  Against 1024
    // workgroups that stay, the whole combine: 300 tokens of hidden 7168 28.4 -> 26.3 us, 600 44.1 -> 40.5, 900 61.1 ->
    // 56.1, 1020 of 4096 42.6 -> 40.7, 2000 of 5120 at top-4 51.0 -> 46.1.
    if (send_blocks > 16384) send_blocks = 16384;
    if (recv_blocks + send_blocks == 0) return 0;
    const size_t lds = size_t(sa.num_local_experts) * sizeof(int32_t);
    // rows returned (read + written) plus rows gathered: past what the caches hold, stream.  Beside more
    // than kLargeBatchRows rows it always pays (11946 of 4 KB, 61.2 -> 57.5 us a step).
    const bool returns_rows = combine_send_slots != nullptr;
    const int64_t traffic = ((returns_rows ? 2 * rows : 0) + int64_t(num_tokens) * num_topk) * hidden * 2;
    const int64_t gather_streams = returns_rows ? kGatherStreamBytes : kGatherAloneStreamBytes;
#define DEEPEP_LAUNCH_FUSED(KERNEL) \
    launch(KERNEL, dim3(unsigned(recv_blocks + send_blocks)), 256, lds, reinterpret_cast<hipStream_t>(stream), sa, ra, int(recv_blocks))
    if (large || traffic > stream_bytes()) DEEPEP_LAUNCH_FUSED(ll_combine_fused_past_caches_kernel);
    else if (traffic > gather_streams) DEEPEP_LAUNCH_FUSED((ll_combine_fused_kernel<true, false>));
    else if (recv_blocks + send_blocks <= kWorkgroupsAtOnce) DEEPEP_LAUNCH_FUSED((ll_combine_fused_kernel<false, true>));
    else DEEPEP_LAUNCH_FUSED((ll_combine_fused_kernel<false, false>));
#undef DEEPEP_LAUNCH_FUSED
    EP_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
