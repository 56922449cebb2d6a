// Host-side error plumbing and device helpers shared by every kernel file.
// gfx950 only: 64-lane wavefronts, DPP lane exchange, hardware OCP-FP8 and
// BF16 pack conversions.
#pragma once
#include <cstdlib>

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace deepep {

// ---------------------------------------------------------------------
// Host errors.  Message format follows the reference's EPException
// (csrc/kernels/exception.cuh:12-22): "Failed: <kind> error <file>:<line> '<what>'".
// ---------------------------------------------------------------------
void set_error(const char* kind, const char* file, int line, const char* what);
void clear_error();

#define EP_HOST_ASSERT(cond)                                                      \
    do {                                                                          \
        if (!(cond)) {                                                            \
            ::deepep::set_error("Assertion", __FILE_NAME__, __LINE__, #cond);     \
            return 1;                                                             \
        }                                                                         \
    } while (0)

#define EP_HIP_CHECK(cmd)                                                                   \
    do {                                                                                    \
        hipError_t e_ = (cmd);                                                              \
        if (e_ != hipSuccess) {                                                             \
            ::deepep::set_error("HIP", __FILE_NAME__, __LINE__, hipGetErrorString(e_));     \
            return 2;                                                                       \
        }                                                                                   \
    } while (0)

// launch(kernel, ..., ...) by the call it stands for.  The launch syntax hands the configuration to the runtime and takes it
// back before that call, and its outcome has to be asked for: 2.52 us of host time a launch against 2.32.  What went
// wrong is the thread's until EP_LAUNCH_CHECK takes it.
inline thread_local hipError_t launch_error = hipSuccess;
inline hipError_t take_launch_error() {
    const hipError_t e = launch_error;
    launch_error = hipSuccess;
    return e;
}
template <typename T>
struct Same {
    typedef T type;
};
template <typename... P>
inline void launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                   typename Same<P>::type... args) {
    void* pointers[] = {&args...};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, lds, stream);
    if (e == hipSuccess) return;
    launch_error = e;
    (void)hipGetLastError();  // reported here and not by whoever asks next
}
#define EP_LAUNCH_CHECK() EP_HIP_CHECK(::deepep::take_launch_error())

// Row formats; values are part of the C ABI.
enum RowFormat : int { kRowBF16 = 0, kRowFP8 = 1, kRowFP8Pow2 = 2, kRowFP8UE8M0 = 3 };

// Hook for a timing build: a harness that wants per-phase timestamps defines DEEPEP_PHASE(i)
// before including the kernels; the library compiles it away.
#ifndef DEEPEP_PHASE
#define DEEPEP_PHASE(i)
#endif

constexpr int kWave = 64;
constexpr int kGroup = 128;        // channels per FP8 scale group
constexpr int kRowTailBytes = 16;  // {src_token, topk_slot, src_rank, local expert}

__host__ __device__ inline int64_t align16(int64_t v) { return (v + 15) & ~int64_t(15); }

__host__ __device__ inline int64_t row_data_bytes(int hidden, int fmt) {
    return fmt == kRowBF16 ? int64_t(hidden) * 2 : int64_t(hidden);
}
__host__ __device__ inline int64_t row_scale_bytes(int hidden, int fmt) {
    if (fmt == kRowBF16) return 0;
    const int g = hidden / kGroup;
    return fmt == kRowFP8UE8M0 ? g : int64_t(g) * 4;
}
// Payload of a staged row: [data | pad16][scales | pad16][tail], what the reference's cooperative send
// calls its stride (csrc/kernels/coop_dispatch_send.cu:73-75).
__host__ __device__ inline int64_t row_payload_bytes(int hidden, int fmt) {
    return align16(row_data_bytes(hidden, fmt)) + align16(row_scale_bytes(hidden, fmt)) + kRowTailBytes;
}
// Distance between staged rows: the payload rounded up to whole 128-byte cache lines, so that a row
// never shares a line with its neighbour.  When the rows come from HBM rather than from the caches
// the send kernel and the receive copy run about 4 % faster than at the bare payload size.
constexpr int kRowAlign = 128;
__host__ __device__ inline int64_t row_stride_bytes(int hidden, int fmt) {
    return (row_payload_bytes(hidden, fmt) + kRowAlign - 1) / kRowAlign * kRowAlign;
}

// ---------------------------------------------------------------------
// Device helpers
// ---------------------------------------------------------------------
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// Wave index inside the workgroup as a scalar, so everything derived from it
// stays in SGPRs and row addresses become scalar loads.
__device__ __forceinline__ int wave_in_block() { return __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6); }

// Threads of the workgroup, as a scalar.  No launch here has a partial workgroup, which blockDim.x allows for: where the
// compiler does not see that it need not, that is a vector load, waited for, ahead of everything else a kernel does.
__device__ __forceinline__ int block_threads() { return int(__builtin_amdgcn_workgroup_size_x()); }

// Stores through a pointer the compiler cannot prove to be global memory (one rebuilt from
// integers, say) are emitted as flat stores, which also tick the LDS counter; these say "global".
typedef __attribute__((address_space(1))) u32x4 global_u32x4;
typedef __attribute__((address_space(1))) uint32_t global_u32;
typedef __attribute__((address_space(1))) uint8_t global_u8;
__device__ __forceinline__ void store_global(uint8_t* p, u32x4 v) { *(global_u32x4*)(p) = v; }
__device__ __forceinline__ void store_global(uint8_t* p, uint32_t v) { *(global_u32*)(p) = v; }
__device__ __forceinline__ u32x4 load_global_u32x4(const uint8_t* p) { return *(const global_u32x4*)(p); }
__device__ __forceinline__ void store_global_byte(uint8_t* p, uint8_t v) { *(global_u8*)(p) = v; }

// Streaming variants for kernels whose traffic exceeds what the caches hold: the non-temporal hint
// keeps lines that will not be touched again from displacing others.  On this GPU a plain device
// copy of 512 MiB runs at 6.1 TB/s with ordinary accesses and 6.6 TB/s with these; eight gathered
// loads in flight per lane read at 6.2 against 7.0 TB/s.  kStream == false is the ordinary access.
template <bool kStream>
__device__ __forceinline__ u32x4 load_u32x4(const uint8_t* p) {
    if constexpr (kStream) return __builtin_nontemporal_load((const global_u32x4*)(p));
    else return *(const global_u32x4*)(p);
}
template <bool kStream>
__device__ __forceinline__ void store_u32x4(uint8_t* p, u32x4 v) {
    if constexpr (kStream) __builtin_nontemporal_store(v, (global_u32x4*)(p));
    else *(global_u32x4*)(p) = v;
}
// Scalar values that have been asked for and must all be there from here on: their loads go out together, in front of
// this, where the compiler would put each behind the branch that first uses it (a trip to memory each).
__device__ __forceinline__ void await_scalars(uint32_t& a, uint32_t& b, uint32_t& c) {
    asm volatile("" : "+s"(a), "+s"(b), "+s"(c));
}
__device__ __forceinline__ void await_scalars(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    asm volatile("" : "+s"(a), "+s"(b), "+s"(c), "+s"(d));
}

// A row as a buffer: its address is the wave's, so a lane brings 32 bits of offset, and lanes past its end read zeros
// and store nothing without a branch.  The row kernels' waves live for one or two trips to memory, so what stands in
// front of the first one counts.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const uint8_t* row, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(row), 0, bytes, 0x00020000);
}
template <bool kStream>
__device__ __forceinline__ u32x4 load_row_u32x4(__amdgpu_buffer_rsrc_t row, int offset) {
    return __builtin_amdgcn_raw_buffer_load_b128(row, offset, 0, kStream ? 2 : 0);  // 2: the non-temporal hint
}
template <bool kStream>
__device__ __forceinline__ void store_row_u32x4(__amdgpu_buffer_rsrc_t row, int offset, u32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, row, offset, 0, kStream ? 2 : 0);
}
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }
__device__ __forceinline__ float bf16_lo(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t packed) { return __uint_as_float(packed & 0xffff0000u); }

// The next kRows rows that `live` names, for the 8 channels at byte `off` of each: lane i holds row i's address and
// weight.
// kInTurn: add() widens one row after the other.  Left to itself the compiler widens all of them ahead of the sums, 32
// registers more than the rows hold (ll_combine_recv_kernel 78 against 50, ll_combine_fused_kernel 76 against 57), and six
// waves fit a SIMD instead of eight.
template <int kRows>
struct RowsInFlight {
    u32x4 v[kRows];
    float w[kRows];
    template <bool kStream, bool kWeighted>
    __device__ __forceinline__ void load(uint64_t address, float weight, uint64_t& live, int off, int row_bytes) {
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const int k = __builtin_ctzll(live);
            live &= ~(uint64_t(1) << k);
            const uint32_t lo = __builtin_amdgcn_readlane(int(uint32_t(address)), k);
            const uint32_t hi = __builtin_amdgcn_readlane(int(uint32_t(address >> 32)), k);
            if constexpr (kWeighted) w[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), k));
            const uint8_t* row = reinterpret_cast<const uint8_t*>((uint64_t(hi) << 32) | lo);
            v[u] = load_row_u32x4<kStream>(row_buffer(row, row_bytes), off);
        }
    }
    template <bool kInTurn, bool kWeighted>
    __device__ __forceinline__ void add(float (&acc)[8]) const {
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (kWeighted) {
                    acc[2 * i] = __builtin_fmaf(bf16_lo(v[u][i]), w[u], acc[2 * i]);
                    acc[2 * i + 1] = __builtin_fmaf(bf16_hi(v[u][i]), w[u], acc[2 * i + 1]);
                } else {
                    acc[2 * i] += bf16_lo(v[u][i]), acc[2 * i + 1] += bf16_hi(v[u][i]);
                }
            }
            if constexpr (kInTurn) __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// acc += weight * row (or row) over the rows that `live` names, in ascending order.  Eight rows are in flight, then what
// is left of eight together; without a branch for each row, which costs a wave as much as the row's arithmetic.
template <bool kStream, bool kWeighted, bool kInTurn>
__device__ __forceinline__ void add_rows(uint64_t address, float weight, uint64_t live, int off, int row_bytes,
                                         float (&acc)[8]) {
    int n = __popcll(live);
    for (; n >= 8; n -= 8) {
        RowsInFlight<8> rows;
        rows.load<kStream, kWeighted>(address, weight, live, off, row_bytes);
        __builtin_amdgcn_sched_barrier(0);  // no row's arithmetic, and so its wait, in front of another's load
        rows.add<kInTurn, kWeighted>(acc);
    }
    RowsInFlight<4> four;
    RowsInFlight<2> two;
    RowsInFlight<1> one;
    if ((n & 4) != 0) four.load<kStream, kWeighted>(address, weight, live, off, row_bytes);
    if ((n & 2) != 0) two.load<kStream, kWeighted>(address, weight, live, off, row_bytes);
    if ((n & 1) != 0) one.load<kStream, kWeighted>(address, weight, live, off, row_bytes);
    __builtin_amdgcn_sched_barrier(0);
    if ((n & 4) != 0) four.add<kInTurn, kWeighted>(acc);
    if ((n & 2) != 0) two.add<kInTurn, kWeighted>(acc);
    if ((n & 1) != 0) one.add<kInTurn, kWeighted>(acc);
}

// Threads [0, threads) of a workgroup move a row, kVecs vectors of each in flight; wider rows go round.
template <int kVecs, bool kStreamLoad, bool kStreamStore>
__device__ __forceinline__ void block_copy_row(const uint8_t* src, uint8_t* dst, int num_vec, int tid, int threads) {
    const auto from = row_buffer(src, num_vec * 16), to = row_buffer(dst, num_vec * 16);
    int v = 0;
    for (;;) {
        u32x4 r[kVecs];
#pragma unroll
        for (int u = 0; u < kVecs; ++u) r[u] = load_row_u32x4<kStreamLoad>(from, (v + u * threads + tid) * 16);
#pragma unroll
        for (int u = 0; u < kVecs; ++u) store_row_u32x4<kStreamStore>(to, (v + u * threads + tid) * 16, r[u]);
        v += kVecs * threads;
        if (v >= num_vec) break;
    }
}
// Threads that move a row's payload, a vector each, at most `most`: wider rows take whole trips of about equal size.
inline int flat_row_threads(int num_vec, int most) {
    const int trips = (num_vec + most - 1) / most;
    return ((num_vec + trips - 1) / trips + 63) / 64 * 64;
}

// Traffic above which a kernel streams (the memory-side cache holds 256 MB).
inline int64_t stream_bytes() { return int64_t(192) << 20; }
// The dispatch streams from 64 MB of traffic on (its stores: the send side's payload and, in the single launch, the
// received rows): with clean caches the hint makes no difference from 512 to 2560
// tokens, with the caches full of another call's dirty lines the send is 18 to 24 % faster with it and
// the single launch 11 to 16 %.  The staged rows themselves, which a transport has just put there, are read the ordinary
// way.  Dispatch of 700 tokens of hidden 4096 and 1000 of 7168, us, hint on the loads too / not: behind a step on other
// buffers 17.4 / 13.5 and 34.4 / 31.0, behind a read of 512 MB 18.8 / 18.2 and 36.9 / 36.4, on the same buffers 17.2 / 12.6
// and 34.6 / 29.4; behind a write of 512 MB, whose lines the rows then push out, 19.5 / 22.1 and 39.4 / 44.
inline int64_t send_stream_bytes() { return int64_t(64) << 20; }

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every
// outstanding global load and store of the wave, which stalls kernels that keep row loads in
// flight across the barrier; use this one where threads exchange data through LDS alone.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A 64-bit value every lane of the wave holds alike, moved to scalar registers.
__device__ __forceinline__ uint64_t wave_uniform_u64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return (uint64_t(hi) << 32) | lo;
}

__device__ __forceinline__ uint64_t lanes_below(int lane) { return (uint64_t(1) << lane) - 1; }

// Two float32 -> bf16, round to nearest even, NaN kept quiet: one instruction.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    typedef float float2_ __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const float2_ v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// max over the 8 lanes that share one 128-channel group (lanes 8i..8i+7):
// two quad permutes and a half-row mirror, all DPP — no LDS traffic.
__device__ __forceinline__ float max_over_8_lanes(float v) {
    int t;
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false);   // quad_perm [1,0,3,2]
    v = fmaxf(v, __int_as_float(t));
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false);   // quad_perm [2,3,0,1]
    v = fmaxf(v, __int_as_float(t));
    t = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false);  // row_half_mirror
    v = fmaxf(v, __int_as_float(t));
    return v;
}

// Inclusive sum over the wave (lane i gets sum of lanes 0..i), all DPP: a log-step shift-add inside
// each row of 16 lanes, then lane 15 of rows 0 and 2 broadcast into rows 1 and 3, then lane 31 into
// rows 2 and 3.
__device__ __forceinline__ int wave_inclusive_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
    return v;
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) v += __shfl_xor(v, d, kWave);
    return v;
}

// 32-bit integer mixer used by the seeded synthesiser (lowbias32 constants).
__host__ __device__ inline uint32_t mix32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

}  // namespace deepep
