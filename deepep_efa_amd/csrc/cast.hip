// Stand-alone per-token FP8 cast (the dispatch path fuses the same
// arithmetic into its send kernel).  One wave = 8 scale groups of one row.
#include "common.hpp"
#include "quant.hpp"
#include "../../include/deepep_hip.h"

namespace deepep {

// kStream: the rows exceed what the caches are worth spending on (they are read once), so they are loaded
// with the non-temporal hint: 16.5 against 17.5 us at 4096 x 7168 with the rows coming from HBM.  The
// results are stored the ordinary way in either case: whoever packs or sends them next reads them.
// Bound by HBM (5.2 TB/s at 4096 x 7168, 5.9 at 12000: the launch's ramp and drain are the difference) and, where the rows
// fit the caches, by what a wave issues: with 32-bit indices instead of 64-bit ones, whose division alone took a hundred
// instructions, and rows as buffers instead of masks 131 x 7168 2.44 -> 2.28 us, 1000 x 7168 5.16 -> 5.05, 2000 x 5120
// 6.87 -> 6.51, 8000 x 4096 19.1 -> 18.6, 4096 x 7168 17.4 -> 16.9.  Past the caches neither more waves a workgroup nor
// runs of neighbouring rows per XCD give more (16.7 to 17.2, and 43.5 to 44.2 at 12000).
template <int kFmt, bool kStream>
__global__ __launch_bounds__(256) void per_token_cast_kernel(const uint8_t* __restrict__ x, uint32_t num_rows,
                                                             uint32_t num_cols, uint32_t pieces_per_row,
                                                             uint8_t* __restrict__ x_fp8,
                                                             uint8_t* __restrict__ scales) {
    const int lane = lane_id();
    const uint32_t item = blockIdx.x * 4 + wave_in_block();
    if (item >= num_rows * pieces_per_row) return;
    const uint32_t row = item / pieces_per_row, piece = item - row * pieces_per_row;
    const uint32_t groups = num_cols / kGroup, group = piece * 8 + (lane >> 3);
    const auto from = row_buffer(x + uint64_t(row) * (num_cols * 2), num_cols * 2);  // zeros past the row's end
    const u32x4 lo = load_row_u32x4<kStream>(from, piece * 2048 + lane * 32);
    const u32x4 hi = load_row_u32x4<kStream>(from, piece * 2048 + lane * 32 + 16);
    uint32_t scale_bits;
    const u32x4 q = quantise_16<kFmt>(lo, hi, scale_bits);
    store_row_u32x4<false>(row_buffer(x_fp8 + uint64_t(row) * num_cols, num_cols), piece * 1024 + lane * 16, q);
    constexpr int kScaleBytes = kFmt == kRowFP8UE8M0 ? 1 : 4;
    const auto row_scales = row_buffer(scales + uint64_t(row) * (groups * kScaleBytes), groups * kScaleBytes);
    const int at = group < groups && (lane & 7) == 0 ? int(group) * kScaleBytes : 0x7fffffff;
    if constexpr (kFmt == kRowFP8UE8M0)  // 4 exponent bytes per int32, little endian
        __builtin_amdgcn_raw_buffer_store_b8(uint8_t(scale_bits >> 23), row_scales, at, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(scale_bits, row_scales, at, 0, 0);
}

}  // namespace deepep

using namespace deepep;

extern "C" int deepep_per_token_cast_to_fp8(const void* x, int num_rows, int num_cols, int row_format, void* x_fp8,
                                            void* scales, void* stream) {
    clear_error();
    EP_HOST_ASSERT(num_rows >= 0 && num_cols > 0 && num_cols % 128 == 0);
    EP_HOST_ASSERT(row_format == kRowFP8 || row_format == kRowFP8Pow2 || row_format == kRowFP8UE8M0);
    EP_HOST_ASSERT(row_format != kRowFP8UE8M0 || (num_cols / 128) % 4 == 0);
    if (num_rows == 0) return 0;
    EP_HOST_ASSERT(x != nullptr && x_fp8 != nullptr && scales != nullptr);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(x_fp8) & 15) == 0);
    EP_HOST_ASSERT((reinterpret_cast<uintptr_t>(scales) & 3) == 0);
    const int pieces = (num_cols / kGroup + 7) / 8;
    EP_HOST_ASSERT(int64_t(num_rows) * pieces < (int64_t(1) << 32) - 8);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const uint8_t* xb = reinterpret_cast<const uint8_t*>(x);
    uint8_t* qb = reinterpret_cast<uint8_t*>(x_fp8);
    uint8_t* sb = reinterpret_cast<uint8_t*>(scales);
    const bool streams = int64_t(num_rows) * num_cols * 3 > send_stream_bytes();
    const unsigned blocks = unsigned((int64_t(num_rows) * pieces + 3) / 4);
#define DEEPEP_LAUNCH_CAST(FMT)                                                                                  \
    do {                                                                                                         \
        if (streams)                                                                                             \
            launch(per_token_cast_kernel<FMT, true>, blocks, 256, 0, s, xb, num_rows, num_cols, pieces, qb, sb);  \
        else                                                                                                     \
            launch(per_token_cast_kernel<FMT, false>, blocks, 256, 0, s, xb, num_rows, num_cols, pieces, qb, sb); \
    } while (0)
    switch (row_format) {
        case kRowFP8: DEEPEP_LAUNCH_CAST(kRowFP8); break;
        case kRowFP8Pow2: DEEPEP_LAUNCH_CAST(kRowFP8Pow2); break;
        default: DEEPEP_LAUNCH_CAST(kRowFP8UE8M0); break;
    }
#undef DEEPEP_LAUNCH_CAST
    EP_LAUNCH_CHECK();
    return 0;
}
