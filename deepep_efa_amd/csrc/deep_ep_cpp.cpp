// deep_ep_cpp — pybind11 host module with the reference's Python-visible surface for the
// dispatch/combine hot path (reference bindings: csrc/deep_ep.cpp:4310-4357,4440-4476).
//
// It owns tensors, checks arguments the way the reference's host code does
// (EP_HOST_ASSERT -> "Failed: Assertion error file:line 'cond'"), hands HIP
// streams around, and calls the C ABI of libdeepep_hip.so for every kernel.
// There is no device code in this file and no CPU fallback: a missing or
// failing HIP library is an exception.
#include <torch/extension.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <pybind11/functional.h>

#include <algorithm>
#include <chrono>
#include <atomic>
#include <functional>
#include <memory>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "../../include/deepep_hip.h"
#include "event.hpp"

namespace deep_ep {

// PyTorch-ROCm tags its HIP streams with the CUDA device type; events and tensors expect that tag.
using HostStream = c10::hip::HIPStreamMasqueradingAsCUDA;
using topk_idx_t = int64_t;  // reference: csrc/kernels/configs.cuh:66-72 (TOPK_IDX_BITS = 64)
constexpr int kNumMaxNvlPeers = 8;            // reference: NUM_MAX_NVL_PEERS, csrc/kernels/configs.cuh:3
constexpr int kNumBufferAlignmentBytes = 128;  // reference: csrc/kernels/configs.cuh:7
constexpr int kSourceMetaBytes = 8;            // reference: internode::get_source_meta_bytes()

#define EP_HOST_ASSERT(cond)                                                          \
    do {                                                                              \
        if (!(cond)) throw ::deep_ep::EPException("Assertion", "deep_ep_cpp.cpp", __LINE__, #cond); \
    } while (0)

// A failed C-ABI call already carries an EPException-shaped message.
static void abi_check(int rc) {
    if (rc != 0) throw EPException(std::string(deepep_last_error()));
}

static hipStream_t current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

template <typename T>
static T align_up(T a, T b) {
    return (a + b - 1) / b * b;
}

// torch::empty without the dispatcher in front of the caching allocator, which is most of its 1.2 us.
static torch::Tensor empty_on(const torch::Device& device, at::IntArrayRef sizes, torch::ScalarType type) {
    return torch::Tensor(at::detail::empty_cuda(sizes, type, device, std::nullopt));
}

// The first n rows of a contiguous tensor, made without the dispatcher (narrow() takes 0.8 us).
static torch::Tensor leading_rows(const torch::Tensor& t, int64_t n) {
    auto rows = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(t.storage()), t.key_set(), t.dtype());
    c10::SmallVector<int64_t, 4> sizes(t.sizes().begin(), t.sizes().end());
    sizes[0] = n;
    rows.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
    rows.unsafeGetTensorImpl()->set_storage_offset(t.storage_offset());
    return rows;
}

// Several results of one call in one allocation.  A torch::empty costs the host 1.2 us and a tensor over a piece
// of storage that exists 0.1 us, so a call with many small results asks the allocator once.
struct ResultBlock {
    int64_t bytes = 0;
    torch::Tensor block;

    int64_t reserve(int64_t size) {  // a byte offset, on a line of its own
        const int64_t at = bytes;
        bytes += align_up<int64_t>(size, 256);
        return at;
    }
    void allocate(const torch::Device& device) {
        block = empty_on(device, {std::max<int64_t>(bytes, 256)}, torch::kUInt8);
    }
    torch::Tensor take(int64_t at, at::IntArrayRef sizes, torch::ScalarType type) const {
        auto t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(block.storage()), block.key_set(),
                                                          c10::scalarTypeToTypeMeta(type));
        t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
        t.unsafeGetTensorImpl()->set_storage_offset(at / int64_t(c10::elementSize(type)));
        return t;
    }
};

// ---------------------------------------------------------------------------
// Config (reference: csrc/config.hpp:23-105) — arithmetic only.
// ---------------------------------------------------------------------------
struct Config {
    int num_sms;
    int num_max_nvl_chunked_send_tokens;
    int num_max_nvl_chunked_recv_tokens;
    int num_max_rdma_chunked_send_tokens;
    int num_max_rdma_chunked_recv_tokens;

    Config(int num_sms, int nvl_send, int nvl_recv, int rdma_send, int rdma_recv)
        : num_sms(num_sms),
          num_max_nvl_chunked_send_tokens(nvl_send),
          num_max_nvl_chunked_recv_tokens(nvl_recv),
          num_max_rdma_chunked_send_tokens(rdma_send),
          num_max_rdma_chunked_recv_tokens(rdma_recv) {
        EP_HOST_ASSERT(num_sms >= 0);
        EP_HOST_ASSERT(nvl_send > 0 and nvl_recv > 0);
        EP_HOST_ASSERT(nvl_send < nvl_recv);
        EP_HOST_ASSERT(rdma_send > 0 and rdma_recv > 0);
        num_max_rdma_chunked_recv_tokens = align_up<int>(rdma_recv, rdma_send);
        EP_HOST_ASSERT(rdma_send < num_max_rdma_chunked_recv_tokens);
        EP_HOST_ASSERT(rdma_send <= num_max_rdma_chunked_recv_tokens / 2);
    }

    size_t get_nvl_buffer_size_hint(size_t hidden_bytes, int num_ranks) const {
        constexpr size_t kNumMaxTopK = 128, kNumMaxScales = 128;
        EP_HOST_ASSERT(num_ranks < kNumMaxNvlPeers or num_ranks % kNumMaxNvlPeers == 0);
        EP_HOST_ASSERT(num_ranks <= kNumMaxNvlPeers or num_sms % 2 == 0);
        const size_t num_rdma_ranks = std::max(num_ranks / kNumMaxNvlPeers, 1);
        const size_t num_nvl_ranks = std::min(num_ranks, kNumMaxNvlPeers);
        const size_t num_channels = num_sms / 2;
        const size_t recv = num_max_nvl_chunked_recv_tokens;
        size_t num_bytes = 0;
        num_bytes += num_channels * num_nvl_ranks * (2 * num_rdma_ranks + 3) * sizeof(int);
        num_bytes += num_channels * num_nvl_ranks * recv * hidden_bytes;
        num_bytes += num_channels * num_nvl_ranks * recv * kSourceMetaBytes;
        num_bytes += num_channels * num_nvl_ranks * recv * kNumMaxTopK * sizeof(topk_idx_t);
        num_bytes += num_channels * num_nvl_ranks * recv * kNumMaxTopK * sizeof(float);
        num_bytes += num_channels * num_nvl_ranks * recv * kNumMaxScales * sizeof(float);
        return ((num_bytes + 127) / 128) * 128;
    }

    size_t get_rdma_buffer_size_hint(int64_t hidden_bytes, int num_ranks) const {
        if (num_ranks <= kNumMaxNvlPeers) return 0;
        constexpr size_t kNumMaxTopK = 128, kNumMaxScales = 128;
        EP_HOST_ASSERT(num_ranks % kNumMaxNvlPeers == 0);
        EP_HOST_ASSERT(num_sms % 2 == 0);
        const size_t num_rdma_ranks = num_ranks / kNumMaxNvlPeers;
        const size_t num_channels = num_sms / 2;
        const size_t recv = num_max_rdma_chunked_recv_tokens;
        size_t num_bytes = 0;
        num_bytes += num_channels * num_rdma_ranks * (kNumMaxNvlPeers * 2 + 2) * 2 * sizeof(int);
        num_bytes += num_channels * num_rdma_ranks * recv * size_t(hidden_bytes) * 2;
        num_bytes += num_channels * num_rdma_ranks * recv * kSourceMetaBytes * 2;
        num_bytes += num_channels * num_rdma_ranks * recv * kNumMaxTopK * sizeof(topk_idx_t) * 2;
        num_bytes += num_channels * num_rdma_ranks * recv * kNumMaxTopK * sizeof(float) * 2;
        num_bytes += num_channels * num_rdma_ranks * recv * kNumMaxScales * sizeof(float) * 2;
        num_bytes += num_channels * num_rdma_ranks * recv * 16 * 2;
        return ((num_bytes + 127) / 128) * 128;
    }
};

static size_t get_low_latency_rdma_size_hint(int num_max_dispatch_tokens_per_rank, int hidden, int num_ranks,
                                             int num_experts) {
    return deepep_get_low_latency_rdma_size_hint(num_max_dispatch_tokens_per_rank, hidden, num_ranks, num_experts);
}

// ---------------------------------------------------------------------------
// EventHandle (reference: csrc/event.hpp:9-25)
// ---------------------------------------------------------------------------
struct EventHandle {
    std::shared_ptr<DeviceEvent> event;

    EventHandle() : EventHandle(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA()) {}
    explicit EventHandle(const HostStream& stream, DeviceEvent::Scope scope = DeviceEvent::kSystem)
        : event(std::make_shared<DeviceEvent>(int(stream.device_index()), stream.stream(), scope)) {}
    void stream_wait_for(const HostStream& waiter) const { event->wait_on(int(waiter.device_index()), waiter.stream()); }
    void current_stream_wait() const { stream_wait_for(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA()); }
};

static void stream_wait(const HostStream& waiter, const HostStream& other) {
    EP_HOST_ASSERT(waiter.id() != other.id());
    torch::Event ev(torch::kCUDA);
    ev.record(other);
    waiter.unwrap().wait(ev);
}

static void stream_wait(const HostStream& waiter, const EventHandle& event) { event.stream_wait_for(waiter); }

// ---------------------------------------------------------------------------
// Low-latency tensors of one shape (reference: the Python-side cache of
// deep_ep/buffer.py:1623-1813; nothing here is cleared per call)
// ---------------------------------------------------------------------------
struct LowLatencyCache {
    int max_tokens = 0, hidden = 0, num_topk = 0, num_experts = 0, row_format = -1;
    torch::Tensor recv_staging, recv_count, send_slots, send_count, pair_slot, workspace, segment_workspace;
    torch::Tensor packed_recv_x, packed_recv_scales, packed_recv_count, packed_recv_src_info, packed_recv_layout_range;
    torch::Tensor combine_staging, combine_send_slots, combined_x;
    bool dispatched = false;
    // What Buffer.low_latency_dispatch returns of it, as the Python objects: ((recv_x, scales) or recv_x, the handle)
    pybind11::object recv_result, handle_result;
};

static int row_format_of(bool use_fp8, bool round_scale, bool use_ue8m0) {
    if (!use_fp8) return DEEPEP_ROW_BF16;
    if (use_ue8m0) return DEEPEP_ROW_FP8_UE8M0;
    return round_scale ? DEEPEP_ROW_FP8_POW2 : DEEPEP_ROW_FP8;
}

// Row-count words (Buffer::observed) of buffers dropped without destroy().  Kernels may still store to them, and the
// garbage collector may drop a buffer during a capture, where nothing can be waited for: such words stay what they
// are and go to the next buffer of the device, for which a late count is a poor hint and no more.  So there are
// never more of them than buffers were alive at a time.
struct RetiredWords {
    std::mutex mutex;
    std::vector<std::pair<int, at::DataPtr>> words;

    static RetiredWords& all() {
        static auto* const the = new RetiredWords;  // never destroyed: the allocator may be gone by then
        return *the;
    }
    static void put(int device, at::DataPtr word) {
        const std::lock_guard<std::mutex> lock(all().mutex);
        all().words.emplace_back(device, std::move(word));
    }
    static at::DataPtr take(int device) {
        const std::lock_guard<std::mutex> lock(all().mutex);
        auto& words = all().words;
        for (auto it = words.begin(); it != words.end(); ++it) {
            if (it->first != device) continue;
            at::DataPtr word = std::move(it->second);
            words.erase(it);
            return word;
        }
        return {};
    }
};

// ---------------------------------------------------------------------------
// Buffer (reference: csrc/deep_ep.hpp:60-707, csrc/deep_ep.cpp:206-581)
// One process, one GPU.  `num_ranks`/`rank` describe the expert-parallel world
// this GPU plays a part in; the other ranks exist only as tensors handed to
// loopback_set_world().
// ---------------------------------------------------------------------------
struct Buffer {
    int rank, num_ranks, rdma_rank, nvl_rank, num_rdma_ranks, num_nvl_ranks;
    int64_t num_nvl_bytes, num_rdma_bytes;
    bool low_latency_mode, explicitly_destroy, enable_shrink;
    bool available = false, destroyed = false;
    int device_id = 0;
    HostStream comm_stream;
    torch::Tensor nvl_buffer, rdma_buffer, mask_status;
    std::unordered_map<int64_t, torch::Tensor> layout_workspaces;  // one per stream that has run the layout kernel
    static constexpr size_t kMaxLayoutWorkspaces = 8;
    LowLatencyCache ll;
    std::vector<torch::Tensor> combine_input_buffers;
    int combine_buffer_idx = 0;
    // What the last two dispatches that have run received, stored there in turn by their kernels as
    // (tokens << 32) | rows: the next call is sized by them.  Under skewed routing a rank can receive many times
    // num_tokens * num_topk rows, and kernels sized for a balanced world walk such a batch in a slow loop.
    at::DataPtr observed_memory;
    std::atomic<uint64_t>* observed = nullptr;  // [2]
    unsigned num_reporting = 0;
    // loopback world
    std::optional<torch::Tensor> world_x, world_topk_idx;
    torch::Tensor ranks_below, ranks_above, peer_workspace;
    int combine_peer_mode = 0;
    uint32_t combine_peer_seed = 0;

    Buffer(int rank, int num_ranks, int64_t num_nvl_bytes, int64_t num_rdma_bytes, bool low_latency_mode,
           bool explicitly_destroy, bool enable_shrink, bool use_fabric)
        : rank(rank),
          num_ranks(num_ranks),
          num_nvl_bytes(num_nvl_bytes),
          num_rdma_bytes(num_rdma_bytes),
          low_latency_mode(low_latency_mode),
          explicitly_destroy(explicitly_destroy),
          enable_shrink(enable_shrink),
          comm_stream(c10::hip::getStreamFromPoolMasqueradingAsCUDA(false)) {  // default priority
        (void)use_fabric;
        EP_HOST_ASSERT(num_ranks > 0 and 0 <= rank and rank < num_ranks);
        EP_HOST_ASSERT(num_nvl_bytes % kNumBufferAlignmentBytes == 0 and num_rdma_bytes % kNumBufferAlignmentBytes == 0);
        EP_HOST_ASSERT(num_ranks <= kNumMaxNvlPeers or num_ranks % kNumMaxNvlPeers == 0 or low_latency_mode);
        rdma_rank = rank / kNumMaxNvlPeers;
        nvl_rank = rank % kNumMaxNvlPeers;
        num_rdma_ranks = std::max(1, num_ranks / kNumMaxNvlPeers);
        num_nvl_ranks = std::min(num_ranks, kNumMaxNvlPeers);
        device_id = c10::hip::current_device();
    }

    ~Buffer() noexcept(false) {
        if (!explicitly_destroy) {
            destroy();
        } else if (!destroyed) {
            if (observed != nullptr) RetiredWords::put(device_id, std::move(observed_memory));
            printf("WARNING: destroy() was not called before DeepEP buffer destruction, which can leak resources.\n");
            fflush(stdout);
        }
    }

    bool is_available() const { return available; }
    bool is_internode_available() const { return is_available() and num_ranks > kNumMaxNvlPeers; }
    int get_num_rdma_ranks() const { return num_rdma_ranks; }
    int get_rdma_rank() const { return rdma_rank; }
    int get_root_rdma_rank(bool global) const { return global ? nvl_rank : 0; }
    int get_local_device_id() const { return device_id; }
    pybind11::bytearray get_local_ipc_handle() const { return pybind11::bytearray(std::string(64, '\0')); }
    c10::Stream get_comm_stream() const { return comm_stream.unwrap(); }

    // One GPU: nothing to open on peers; the call only marks the buffer usable.
    void sync(const std::vector<int>& device_ids, const std::vector<std::optional<pybind11::bytearray>>& handles,
              const std::optional<pybind11::bytearray>& root_unique_id) {
        (void)handles;
        (void)root_unique_id;
        EP_HOST_ASSERT(not is_available());
        EP_HOST_ASSERT(device_ids.empty() or static_cast<int>(device_ids.size()) == num_ranks or device_ids.size() == 1);
        available = true;
    }

    // The host allocator does not know of the kernels that store to the pinned word: it gets the word back when
    // none is left in flight, or its next owner would find a row count in it.
    void release_observed() {
        if (observed == nullptr) return;
        const c10::DeviceGuard on_device(torch::Device(torch::kCUDA, static_cast<c10::DeviceIndex>(device_id)));
        (void)hipDeviceSynchronize();
        observed = nullptr;
        observed_memory.clear();
    }

    void destroy() {
        if (destroyed) return;
        if (available) (void)hipDeviceSynchronize();
        release_observed();
        nvl_buffer = torch::Tensor();
        rdma_buffer = torch::Tensor();
        layout_workspaces.clear();
        ll = LowLatencyCache();
        combine_input_buffers.clear();
        world_x.reset();
        world_topk_idx.reset();
        peer_workspace = torch::Tensor();
        destroyed = true;
        available = false;
    }

    torch::Tensor get_local_buffer_tensor(const pybind11::object& dtype, int64_t offset, bool use_rdma_buffer) {
        torch::ScalarType casted = torch::python::detail::py_object_to_dtype(dtype);
        const int64_t element_bytes = static_cast<int64_t>(elementSize(casted));
        torch::Tensor& base = use_rdma_buffer ? rdma_buffer : nvl_buffer;
        const int64_t num_bytes = use_rdma_buffer ? num_rdma_bytes : num_nvl_bytes;
        if (!base.defined())  // allocated on first use; valid until destroy()
            base = torch::empty({std::max<int64_t>(num_bytes, 16)}, torch::dtype(torch::kUInt8).device(torch::kCUDA));
        EP_HOST_ASSERT(offset >= 0 and offset <= num_bytes);
        auto bytes = base.narrow(0, offset, ((num_bytes - offset) / element_bytes) * element_bytes);
        return bytes.view(casted);
    }

    // -- layout ---------------------------------------------------------------
    std::tuple<torch::Tensor, std::optional<torch::Tensor>, torch::Tensor, torch::Tensor, std::optional<EventHandle>>
    get_dispatch_layout(const torch::Tensor& topk_idx, int num_experts, std::optional<EventHandle>& previous_event,
                        bool async, bool allocate_on_comm_stream) {
        EP_HOST_ASSERT(topk_idx.dim() == 2);
        EP_HOST_ASSERT(topk_idx.is_contiguous());
        EP_HOST_ASSERT(topk_idx.is_cuda() and topk_idx.scalar_type() == torch::kInt64);
        EP_HOST_ASSERT(num_experts > 0);

        auto compute_stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA();
        // A synchronous call with nothing to wait for is ordered on the caller's stream either way: the
        // reference moves the work to its communication stream and back through two events
        // (csrc/deep_ep.cpp:526-537,559-574), which on this GPU costs more than the kernels (27 us against 7);
        // here such a call runs on the caller's stream directly.  Every other form keeps the hand-off.
        const bool in_place = not async and not previous_event.has_value() and not allocate_on_comm_stream;
        auto work_stream = in_place ? compute_stream : comm_stream;
        if (allocate_on_comm_stream) {
            EP_HOST_ASSERT(previous_event.has_value() and async);
            c10::hip::setCurrentHIPStreamMasqueradingAsCUDA(comm_stream);
        }
        if (previous_event.has_value())
            stream_wait(comm_stream, previous_event.value());
        else if (not in_place)
            stream_wait(comm_stream, compute_stream);

        const int num_tokens = static_cast<int>(topk_idx.size(0)), num_topk = static_cast<int>(topk_idx.size(1));
        ResultBlock b;
        const int64_t rank_at = b.reserve(4 * num_ranks), rdma_at = b.reserve(4 * num_rdma_ranks);
        const int64_t expert_at = b.reserve(4 * num_experts), member_at = b.reserve(int64_t(num_tokens) * num_ranks);
        b.allocate(torch::kCUDA);
        auto num_tokens_per_rank = b.take(rank_at, {num_ranks}, torch::kInt32);
        auto num_tokens_per_rdma_rank = std::optional<torch::Tensor>();
        auto num_tokens_per_expert = b.take(expert_at, {num_experts}, torch::kInt32);
        auto is_token_in_rank = b.take(member_at, {num_tokens, num_ranks}, torch::kBool);
        if (is_internode_available()) num_tokens_per_rdma_rank = b.take(rdma_at, {num_rdma_ranks}, torch::kInt32);

        const int64_t ws_bytes =
            std::max<int64_t>(256, int64_t(deepep_layout_workspace_bytes(num_tokens, num_ranks, num_experts)));
        // the kernel's scratch belongs to the stream the kernel runs on: a call on the buffer's own stream and
        // one on the caller's stream may be in flight together
        if (layout_workspaces.size() >= kMaxLayoutWorkspaces and layout_workspaces.count(int64_t(work_stream.id())) == 0)
            layout_workspaces.clear();  // a caller cycling through streams does not grow the table without bound
        torch::Tensor& layout_workspace = layout_workspaces[int64_t(work_stream.id())];
        if (!layout_workspace.defined() or layout_workspace.numel() < ws_bytes) {
            // allocated with the kernel's stream current, so that the caching allocator ties the block to that
            // stream: a block dropped here (replaced, or the table cleared) is handed out again only to
            // allocations ordered behind the kernels that used it
            c10::hip::HIPStreamGuardMasqueradingAsCUDA on_work_stream(work_stream.unwrap());
            layout_workspace = torch::empty({ws_bytes}, torch::dtype(torch::kUInt8).device(torch::kCUDA));
        }

        abi_check(deepep_get_dispatch_layout(
            topk_idx.data_ptr<int64_t>(), num_tokens, num_topk, num_ranks, num_experts,
            num_tokens_per_rank.data_ptr<int>(),
            num_tokens_per_rdma_rank.has_value() ? num_tokens_per_rdma_rank->data_ptr<int>() : nullptr,
            num_tokens_per_expert.data_ptr<int>(), reinterpret_cast<uint8_t*>(is_token_in_rank.data_ptr<bool>()),
            layout_workspace.data_ptr(), size_t(layout_workspace.numel()), work_stream.stream()));

        std::optional<EventHandle> event;
        if (async) {
            event = EventHandle(comm_stream);
            for (auto& t : {topk_idx, num_tokens_per_rank, num_tokens_per_expert, is_token_in_rank}) {
                t.record_stream(comm_stream);
                if (allocate_on_comm_stream) t.record_stream(compute_stream);
            }
            if (num_tokens_per_rdma_rank.has_value()) {
                num_tokens_per_rdma_rank->record_stream(comm_stream);
                if (allocate_on_comm_stream) num_tokens_per_rdma_rank->record_stream(compute_stream);
            }
        } else if (not in_place) {
            stream_wait(compute_stream, comm_stream);
        }
        if (allocate_on_comm_stream) c10::hip::setCurrentHIPStreamMasqueradingAsCUDA(compute_stream);
        return {num_tokens_per_rank, num_tokens_per_rdma_rank, num_tokens_per_expert, is_token_in_rank, event};
    }

    // -- loopback world ---------------------------------------------------------
    void loopback_set_world(const torch::Tensor& x_all, const torch::Tensor& topk_idx_all) {
        EP_HOST_ASSERT(x_all.dim() == 3 and x_all.is_contiguous() and x_all.is_cuda());
        EP_HOST_ASSERT(x_all.scalar_type() == torch::kBFloat16);
        EP_HOST_ASSERT(topk_idx_all.dim() == 3 and topk_idx_all.is_contiguous() and topk_idx_all.is_cuda());
        EP_HOST_ASSERT(topk_idx_all.scalar_type() == torch::kInt64);
        EP_HOST_ASSERT(x_all.size(0) == num_ranks and topk_idx_all.size(0) == num_ranks);
        EP_HOST_ASSERT(x_all.size(1) == topk_idx_all.size(1));
        world_x = x_all;
        world_topk_idx = topk_idx_all;
        auto i32 = torch::dtype(torch::kInt32).device(torch::kCUDA);
        ranks_below = torch::arange(0, rank, i32);
        ranks_above = torch::arange(rank + 1, num_ranks, i32);
    }

    void loopback_clear_world() {
        world_x.reset();
        world_topk_idx.reset();
    }

    void loopback_synthesise(int num_tokens, int hidden, int num_topk, int num_experts, const torch::Tensor& expert_cdf,
                             int outlier_period, int64_t seed) {
        EP_HOST_ASSERT(expert_cdf.is_cuda() and expert_cdf.is_contiguous() and expert_cdf.numel() == num_experts);
        EP_HOST_ASSERT(expert_cdf.element_size() == 4);
        auto ranks = torch::arange(0, num_ranks, torch::dtype(torch::kInt32).device(torch::kCUDA));
        auto topk = torch::empty({num_ranks, num_tokens, num_topk}, torch::dtype(torch::kInt64).device(torch::kCUDA));
        auto x = torch::empty({num_ranks, num_tokens, hidden}, torch::dtype(torch::kBFloat16).device(torch::kCUDA));
        abi_check(deepep_synth_topk_idx(reinterpret_cast<const uint32_t*>(expert_cdf.data_ptr()), ranks.data_ptr<int>(),
                                        num_ranks, num_tokens, num_topk, num_experts, uint32_t(seed),
                                        topk.data_ptr<int64_t>(), current_stream()));
        abi_check(deepep_synth_bf16_rows(x.data_ptr(), int64_t(num_ranks) * num_tokens, hidden, int64_t(hidden) * 2,
                                         nullptr, 0, uint32_t(seed), outlier_period, current_stream()));
        loopback_set_world(x, topk);
    }

    std::tuple<torch::Tensor, torch::Tensor> loopback_own_inputs() const {
        EP_HOST_ASSERT(world_x.has_value());
        return {world_x->select(0, rank), world_topk_idx->select(0, rank)};
    }

    std::tuple<torch::Tensor, torch::Tensor> loopback_world() const {
        EP_HOST_ASSERT(world_x.has_value());
        return {*world_x, *world_topk_idx};
    }

    void loopback_set_combine_mode(int mode, int64_t seed) {
        EP_HOST_ASSERT(mode == 0 or mode == 1);
        combine_peer_mode = mode;
        combine_peer_seed = uint32_t(seed);
    }

    // -- low latency ------------------------------------------------------------
    LowLatencyCache& get_ll_cache(int max_tokens, int hidden, int num_topk, int num_experts, int fmt) {
        if (ll.max_tokens == max_tokens and ll.hidden == hidden and ll.num_topk == num_topk and
            ll.num_experts == num_experts and ll.row_format == fmt)
            return ll;
        ll = LowLatencyCache();
        ll.max_tokens = max_tokens, ll.hidden = hidden, ll.num_topk = num_topk, ll.num_experts = num_experts;
        ll.row_format = fmt;
        const int64_t el = num_experts / num_ranks, r = num_ranks, m = max_tokens, e = num_experts, h = hidden;
        const int64_t stride = int64_t(deepep_ll_row_stride(hidden, fmt));
        auto u8 = torch::dtype(torch::kUInt8).device(torch::kCUDA);
        auto i32 = torch::dtype(torch::kInt32).device(torch::kCUDA);
        auto bf16 = torch::dtype(torch::kBFloat16).device(torch::kCUDA);
        ll.recv_staging = torch::empty({el * r * m * stride}, u8);
        ll.recv_count = torch::zeros({el * r}, i32);
        ll.send_slots = torch::empty({e * m * stride}, u8);
        ll.send_count = torch::zeros({e}, i32);
        ll.pair_slot = torch::full({m, num_topk}, -1, i32);
        ll.workspace = torch::empty(
            {std::max<int64_t>(256, int64_t(deepep_ll_dispatch_workspace_bytes(max_tokens, num_topk, num_experts)))}, u8);
        // index + flat-copy scratch, used where more than 8192 rows are expected
        ll.segment_workspace = torch::empty({int64_t(deepep_ll_segment_workspace_bytes(num_experts, max_tokens))}, u8);
        if (fmt == DEEPEP_ROW_BF16) {
            ll.packed_recv_x = torch::empty({el, r * m, h}, bf16);
        } else {
            ll.packed_recv_x = torch::empty({el, r * m, h}, torch::dtype(torch::kFloat8_e4m3fn).device(torch::kCUDA));
            if (fmt == DEEPEP_ROW_FP8_UE8M0)
                ll.packed_recv_scales = torch::empty({el, r * m, h / 512}, i32);
            else
                ll.packed_recv_scales = torch::empty({el, r * m, h / 128}, torch::dtype(torch::kFloat32).device(torch::kCUDA));
        }
        ll.packed_recv_count = torch::zeros({el}, i32);
        ll.packed_recv_src_info = torch::empty({el, r * m}, i32);
        ll.packed_recv_layout_range = torch::zeros({el, r}, torch::dtype(torch::kInt64).device(torch::kCUDA));
        ll.combine_staging = torch::empty({e, m, h}, bf16);
        ll.combine_send_slots = torch::empty({el, r, m, h}, bf16);
        ll.combined_x = torch::empty({m, h}, bf16);
        return ll;
    }

    // Rows a batch of num_tokens probably receives, from what the last two did.
    int64_t rows_expected(int num_tokens, int num_topk, int num_experts, int max_tokens) const {
        if (observed == nullptr) return deepep_ll_expected_rows(num_tokens, num_topk, num_experts, max_tokens, 0);
        return deepep_ll_expected_rows_of_two(num_tokens, num_topk, num_experts, max_tokens,
                                              observed[0].load(std::memory_order_relaxed),
                                              observed[1].load(std::memory_order_relaxed));
    }

    void stage_peer_rows(LowLatencyCache& c) {
        if (!world_x.has_value()) return;
        const int t = static_cast<int>(world_x->size(1)), h = static_cast<int>(world_x->size(2));
        const int k = static_cast<int>(world_topk_idx->size(2));
        EP_HOST_ASSERT(h == c.hidden and k == c.num_topk and t <= c.max_tokens);
        const int64_t per = int64_t(deepep_ll_dispatch_workspace_bytes(t, k, c.num_experts));
        const int64_t need = std::max<int64_t>(256, per * std::max({rank, num_ranks - 1 - rank, 1}));
        if (!peer_workspace.defined() or peer_workspace.numel() < need)
            peer_workspace = torch::empty({need}, torch::dtype(torch::kUInt8).device(torch::kCUDA));
        const torch::Tensor* groups[2] = {&ranks_below, &ranks_above};
        const int first[2] = {0, rank + 1};
        for (int g = 0; g < 2; ++g) {
            const int n = static_cast<int>(groups[g]->numel());
            if (n == 0) continue;
            abi_check(deepep_loopback_dispatch_from_peers(
                world_x->select(0, first[g]).data_ptr(), world_topk_idx->select(0, first[g]).data_ptr<int64_t>(),
                groups[g]->data_ptr<int>(), n, t, h, k, c.num_experts, num_ranks, rank, c.max_tokens, c.row_format,
                c.recv_staging.data_ptr(), c.recv_count.data_ptr<int>(), peer_workspace.data_ptr(),
                size_t(peer_workspace.numel()), current_stream()));
        }
    }

    LowLatencyCache& run_low_latency_dispatch(const torch::Tensor& x, const torch::Tensor& topk_idx,
                                              const torch::Tensor* cumulative_local_expert_recv_stats,
                                              const torch::Tensor* dispatch_wait_recv_cost_stats,
                                              int num_max_dispatch_tokens_per_rank, int num_experts, bool use_fp8,
                                              bool round_scale, bool use_ue8m0) {
        EP_HOST_ASSERT(low_latency_mode);
        // reference checks: csrc/deep_ep.cpp:1674-1693
        EP_HOST_ASSERT(x.dim() == 2 and x.is_contiguous() and x.scalar_type() == torch::kBFloat16);
        EP_HOST_ASSERT(x.is_cuda() and topk_idx.is_cuda());
        EP_HOST_ASSERT(x.size(1) % 16 == 0 and x.size(1) % 128 == 0);
        EP_HOST_ASSERT(topk_idx.dim() == 2 and topk_idx.is_contiguous());
        EP_HOST_ASSERT(x.size(0) == topk_idx.size(0) and x.size(0) <= num_max_dispatch_tokens_per_rank);
        EP_HOST_ASSERT(topk_idx.scalar_type() == torch::kInt64);
        EP_HOST_ASSERT(num_experts % num_ranks == 0);
        EP_HOST_ASSERT(not use_ue8m0 or round_scale);
        EP_HOST_ASSERT(not use_ue8m0 or (x.size(1) / 128) % 4 == 0);
        if (cumulative_local_expert_recv_stats != nullptr) {
            EP_HOST_ASSERT(cumulative_local_expert_recv_stats->scalar_type() == torch::kInt);
            EP_HOST_ASSERT(cumulative_local_expert_recv_stats->dim() == 1 and
                           cumulative_local_expert_recv_stats->is_contiguous());
            EP_HOST_ASSERT(cumulative_local_expert_recv_stats->size(0) == num_experts / num_ranks);
        }
        if (dispatch_wait_recv_cost_stats != nullptr) {
            EP_HOST_ASSERT(dispatch_wait_recv_cost_stats->scalar_type() == torch::kInt64);
            EP_HOST_ASSERT(dispatch_wait_recv_cost_stats->dim() == 1 and dispatch_wait_recv_cost_stats->is_contiguous());
            EP_HOST_ASSERT(dispatch_wait_recv_cost_stats->size(0) == num_ranks);
        }
        const int num_tokens = static_cast<int>(x.size(0)), hidden = static_cast<int>(x.size(1));
        const int num_topk = static_cast<int>(topk_idx.size(1));
        const int fmt = row_format_of(use_fp8, round_scale, use_ue8m0);
        auto& c = get_ll_cache(num_max_dispatch_tokens_per_rank, hidden, num_topk, num_experts, fmt);
        auto stream = current_stream();

        stage_peer_rows(c);  // what the exchange would have delivered
        // a captured call takes the hint but does not report: its replays may outlive the buffer, and a capture is
        // no place to allocate pinned memory
        const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
        if (observed == nullptr and not capturing) {
            observed_memory = RetiredWords::take(device_id);
            if (!observed_memory) observed_memory = at::getHostAllocator(at::kCUDA)->allocate(2 * sizeof(uint64_t));
            observed = static_cast<std::atomic<uint64_t>*>(observed_memory.get());
            for (int i = 0; i < 2; ++i) new (observed + i) std::atomic<uint64_t>(0);
        }
        // send and receive phase in one call (one kernel launch for decode-sized batches)
        abi_check(deepep_ll_dispatch_observed(
            x.data_ptr(), topk_idx.data_ptr<int64_t>(), num_tokens, hidden, num_topk, num_experts, num_ranks, rank,
            num_max_dispatch_tokens_per_rank, fmt, c.recv_staging.data_ptr(), c.recv_count.data_ptr<int>(),
            c.send_slots.data_ptr(), c.send_count.data_ptr<int>(), c.pair_slot.data_ptr<int>(),
            c.packed_recv_x.data_ptr(), c.packed_recv_scales.defined() ? c.packed_recv_scales.data_ptr() : nullptr,
            c.packed_recv_src_info.data_ptr<int>(), c.packed_recv_layout_range.data_ptr<int64_t>(),
            c.packed_recv_count.data_ptr<int>(),
            cumulative_local_expert_recv_stats != nullptr ? cumulative_local_expert_recv_stats->data_ptr<int>() : nullptr,
            rows_expected(num_tokens, num_topk, num_experts, num_max_dispatch_tokens_per_rank), c.workspace.data_ptr(),
            size_t(c.workspace.numel()), c.segment_workspace.data_ptr(), size_t(c.segment_workspace.numel()),
            capturing ? nullptr : reinterpret_cast<uint64_t*>(observed + (num_reporting++ & 1)), stream));
        c.dispatched = true;
        return c;
    }

    std::tuple<torch::Tensor, std::optional<torch::Tensor>, torch::Tensor, torch::Tensor, torch::Tensor,
               std::optional<EventHandle>, std::optional<std::function<void()>>>
    low_latency_dispatch(const torch::Tensor& x, const torch::Tensor& topk_idx,
                         const std::optional<torch::Tensor>& cumulative_local_expert_recv_stats,
                         const std::optional<torch::Tensor>& dispatch_wait_recv_cost_stats,
                         int num_max_dispatch_tokens_per_rank, int num_experts, bool use_fp8, bool round_scale,
                         bool use_ue8m0, bool async, bool return_recv_hook) {
        auto given = [](const std::optional<torch::Tensor>& t) { return t.has_value() ? &t.value() : nullptr; };
        auto& c = run_low_latency_dispatch(x, topk_idx, given(cumulative_local_expert_recv_stats),
                                           given(dispatch_wait_recv_cost_stats), num_max_dispatch_tokens_per_rank,
                                           num_experts, use_fp8, round_scale, use_ue8m0);
        std::optional<EventHandle> event;
        if (async) event = EventHandle();
        std::optional<std::function<void()>> hook;
        if (return_recv_hook) hook = [] {};
        std::optional<torch::Tensor> scales;
        if (c.packed_recv_scales.defined()) scales = c.packed_recv_scales;
        return {c.packed_recv_x, scales, c.packed_recv_count, c.packed_recv_src_info, c.packed_recv_layout_range,
                event, hook};
    }

    torch::Tensor run_low_latency_combine(const torch::Tensor& x, const torch::Tensor& topk_idx,
                                          const torch::Tensor& topk_weights, const torch::Tensor& src_info,
                                          const torch::Tensor& layout_range,
                                          const torch::Tensor* combine_wait_recv_cost_stats,
                                          int num_max_dispatch_tokens_per_rank, int num_experts, bool zero_copy,
                                          const torch::Tensor* out, bool accumulate) {
        // accumulate: the sum starts from what `out` holds (the reference has the flag on its reduce binding,
        // csrc/deep_ep.cpp:3850-3857, kernel csrc/kernels/coop_combine_recv.cuh:174-179)
        EP_HOST_ASSERT(not accumulate or out != nullptr);
        EP_HOST_ASSERT(low_latency_mode);
        // reference checks: csrc/deep_ep.cpp:1816-1837
        EP_HOST_ASSERT(x.dim() == 3 and x.is_contiguous() and x.scalar_type() == torch::kBFloat16);
        EP_HOST_ASSERT(x.size(0) == num_experts / num_ranks);
        EP_HOST_ASSERT(x.size(1) == int64_t(num_ranks) * num_max_dispatch_tokens_per_rank);
        EP_HOST_ASSERT(x.size(2) % 16 == 0 and x.size(2) % 128 == 0);
        EP_HOST_ASSERT(topk_idx.dim() == 2 and topk_idx.is_contiguous());
        EP_HOST_ASSERT(topk_idx.size(0) == topk_weights.size(0) and topk_idx.size(1) == topk_weights.size(1));
        EP_HOST_ASSERT(topk_idx.scalar_type() == torch::kInt64);
        EP_HOST_ASSERT(topk_weights.dim() == 2 and topk_weights.is_contiguous());
        EP_HOST_ASSERT(topk_weights.size(0) <= num_max_dispatch_tokens_per_rank);
        EP_HOST_ASSERT(topk_weights.scalar_type() == torch::kFloat32);
        EP_HOST_ASSERT(src_info.dim() == 2 and src_info.is_contiguous());
        EP_HOST_ASSERT(src_info.scalar_type() == torch::kInt32 and x.size(0) == src_info.size(0));
        EP_HOST_ASSERT(layout_range.dim() == 2 and layout_range.is_contiguous());
        EP_HOST_ASSERT(layout_range.scalar_type() == torch::kInt64);
        EP_HOST_ASSERT(layout_range.size(0) == num_experts / num_ranks and layout_range.size(1) == num_ranks);
        if (combine_wait_recv_cost_stats != nullptr) {
            EP_HOST_ASSERT(combine_wait_recv_cost_stats->scalar_type() == torch::kInt64);
            EP_HOST_ASSERT(combine_wait_recv_cost_stats->dim() == 1 and combine_wait_recv_cost_stats->is_contiguous());
            EP_HOST_ASSERT(combine_wait_recv_cost_stats->size(0) == num_ranks);
        }
        const int hidden = static_cast<int>(x.size(2));
        const int num_topk = static_cast<int>(topk_weights.size(1));
        const int num_combined_tokens = static_cast<int>(topk_weights.size(0));
        // the slots of this rank's own pairs were fixed by the dispatch that produced `handle`
        EP_HOST_ASSERT(ll.dispatched and ll.max_tokens == num_max_dispatch_tokens_per_rank and ll.hidden == hidden and
                       ll.num_topk == num_topk and ll.num_experts == num_experts);
        auto& c = ll;
        auto stream = current_stream();

        const torch::Tensor* src = &x;
        // zero_copy: the caller wrote its expert outputs into the buffer handed out earlier, and that buffer is
        // what the transport sends from (the ranges of layout_range are contiguous in it), so the combine skips
        // the row return -- "the next combine kernel can skip the copying", deep_ep/buffer.py:2831-2852
        if (zero_copy) {
            EP_HOST_ASSERT(!combine_input_buffers.empty() and combine_input_buffers[combine_buffer_idx].defined());
            src = &combine_input_buffers[combine_buffer_idx];
            EP_HOST_ASSERT(src->size(0) == x.size(0) and src->size(1) == x.size(1) and src->size(2) == x.size(2));
        }
        torch::Tensor combined_x;
        if (out != nullptr) {
            EP_HOST_ASSERT(out->dim() == 2 and out->is_contiguous() and out->scalar_type() == torch::kBFloat16);
            EP_HOST_ASSERT(out->size(0) == num_combined_tokens and out->size(1) == hidden);
            combined_x = *out;
        } else {
            combined_x = leading_rows(c.combined_x, num_combined_tokens);
        }

        if (world_x.has_value())  // what the remote experts would have returned
            abi_check(deepep_loopback_combine_from_peers(c.send_slots.data_ptr(), c.send_count.data_ptr<int>(), hidden,
                                                         num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank,
                                                         c.row_format, combine_peer_mode, combine_peer_seed,
                                                         c.combine_staging.data_ptr(), stream));
        // row return and weighted reduce in one call (one kernel launch for decode-sized batches)
        abi_check(deepep_ll_combine(src->data_ptr(), layout_range.data_ptr<int64_t>(), topk_idx.data_ptr<int64_t>(),
                                    topk_weights.data_ptr<float>(), c.pair_slot.data_ptr<int>(), num_combined_tokens,
                                    hidden, num_topk, num_experts, num_ranks, rank, num_max_dispatch_tokens_per_rank,
                                    accumulate ? 1 : 0, c.combine_staging.data_ptr(),
                                    zero_copy ? nullptr : c.combine_send_slots.data_ptr(),
                                    combined_x.data_ptr(),
                                    rows_expected(num_combined_tokens, num_topk, num_experts,
                                                  num_max_dispatch_tokens_per_rank),
                                    c.segment_workspace.data_ptr(), size_t(c.segment_workspace.numel()), stream));

        return combined_x;
    }

    std::tuple<torch::Tensor, std::optional<EventHandle>, std::optional<std::function<void()>>> low_latency_combine(
        const torch::Tensor& x, const torch::Tensor& topk_idx, const torch::Tensor& topk_weights,
        const torch::Tensor& src_info, const torch::Tensor& layout_range,
        const std::optional<torch::Tensor>& combine_wait_recv_cost_stats, int num_max_dispatch_tokens_per_rank,
        int num_experts, bool use_logfmt, bool zero_copy, bool async, bool return_recv_hook,
        const std::optional<torch::Tensor>& out, bool accumulate) {
        (void)use_logfmt;
        auto given = [](const std::optional<torch::Tensor>& t) { return t.has_value() ? &t.value() : nullptr; };
        auto combined_x = run_low_latency_combine(x, topk_idx, topk_weights, src_info, layout_range,
                                                  given(combine_wait_recv_cost_stats), num_max_dispatch_tokens_per_rank,
                                                  num_experts, zero_copy, given(out), accumulate);
        std::optional<EventHandle> event;
        if (async) event = EventHandle();
        std::optional<std::function<void()>> hook;
        if (return_recv_hook) hook = [] {};
        return {combined_x, event, hook};
    }

    torch::Tensor get_next_low_latency_combine_buffer(int num_max_dispatch_tokens_per_rank, int hidden, int num_experts) {
        EP_HOST_ASSERT(low_latency_mode);
        if (combine_input_buffers.empty()) combine_input_buffers.resize(2);
        auto& buf = combine_input_buffers[combine_buffer_idx];
        const int64_t el = num_experts / num_ranks, n = int64_t(num_ranks) * num_max_dispatch_tokens_per_rank;
        if (!buf.defined() or buf.size(0) != el or buf.size(1) != n or buf.size(2) != hidden)
            buf = torch::zeros({el, n, hidden}, torch::dtype(torch::kBFloat16).device(torch::kCUDA));
        return buf;
    }

    void clean_low_latency_buffer(int num_max_dispatch_tokens_per_rank, int hidden, int num_experts) {
        (void)num_max_dispatch_tokens_per_rank;
        (void)hidden;
        (void)num_experts;
        EP_HOST_ASSERT(low_latency_mode);
        combine_buffer_idx = 0;
        for (auto& b : combine_input_buffers)
            if (b.defined()) b.zero_();
        if (ll.recv_count.defined()) ll.recv_count.zero_();
        ll.dispatched = false;
    }

    void ensure_mask() {
        if (!mask_status.defined())
            mask_status = torch::zeros({num_ranks}, torch::dtype(torch::kInt32).device(torch::kCUDA));
    }
    void low_latency_update_mask_buffer(int rank_to_mask, bool mask) {
        EP_HOST_ASSERT(rank_to_mask >= 0 and rank_to_mask < num_ranks);
        ensure_mask();
        mask_status.select(0, rank_to_mask).fill_(mask ? 1 : 0);
    }
    void low_latency_query_mask_buffer(torch::Tensor& out) {
        EP_HOST_ASSERT(out.numel() == num_ranks and out.scalar_type() == torch::kInt32);
        ensure_mask();
        out.copy_(mask_status);
    }
    void low_latency_clean_mask_buffer() {
        if (mask_status.defined()) mask_status.zero_();
    }
};

// ---------------------------------------------------------------------------
// Free functions
// ---------------------------------------------------------------------------
// reference: csrc/kernels/efa_kernels.cu:2281-2327
static std::tuple<torch::Tensor, torch::Tensor> per_token_cast_to_fp8(const torch::Tensor& x, bool round_scale,
                                                                      bool use_ue8m0) {
    EP_HOST_ASSERT(x.dim() == 2 && x.is_contiguous() && x.is_cuda());
    EP_HOST_ASSERT(x.scalar_type() == torch::kBFloat16);
    const int m = static_cast<int>(x.size(0)), n = static_cast<int>(x.size(1));
    EP_HOST_ASSERT(n % 128 == 0);
    EP_HOST_ASSERT(not use_ue8m0 or round_scale);
    const int g = n / 128;
    auto x_fp8 = empty_on(x.device(), {m, n}, torch::kFloat8_e4m3fn);
    torch::Tensor scales;
    if (use_ue8m0) {
        EP_HOST_ASSERT(g % 4 == 0);
        scales = empty_on(x.device(), {m, g / 4}, torch::kInt32);
    } else {
        scales = empty_on(x.device(), {m, g}, torch::kFloat32);
    }
    abi_check(deepep_per_token_cast_to_fp8(x.data_ptr(), m, n, row_format_of(true, round_scale, use_ue8m0),
                                           x_fp8.data_ptr(), scales.data_ptr(), current_stream()));
    return {x_fp8, scales};
}

// Words of pinned memory that the workgroups of a kernel store to when they are done and the host polls.  Reading 8
// bytes back with a copy and a synchronisation takes 16 us of an idle stream (the copy is a kernel of its own); a launch
// and a synchronisation take 11 us, a launch and the poll 6.
class HostWords {
    at::DataPtr memory;
    std::atomic<int64_t>* words;
    int count;
    static constexpr int64_t kUnset = INT64_MIN;

public:
    explicit HostWords(int n) : memory(at::getHostAllocator(at::kCUDA)->allocate(sizeof(int64_t) * size_t(n))), count(n) {
        static_assert(sizeof(std::atomic<int64_t>) == sizeof(int64_t));
        words = static_cast<std::atomic<int64_t>*>(memory.get());
        for (int i = 0; i < n; ++i) new (words + i) std::atomic<int64_t>(kUnset);
    }
    int64_t* device_pointer() const { return reinterpret_cast<int64_t*>(words); }
    // Waits for all words and returns the last; `stream` is the one whose kernel stores them.  A stream that is busy
    // for long is waited for in the ordinary way, which also reports what went wrong on it.
    int64_t wait(hipStream_t stream) const {
        pybind11::gil_scoped_release release;
        const auto began = std::chrono::steady_clock::now();
        int spins = 0;
        for (int i = 0; i < count;) {
            if (words[i].load(std::memory_order_acquire) != kUnset) {
                ++i;
                continue;
            }
            __builtin_ia32_pause();
            if (++spins % 1024 == 0 and std::chrono::steady_clock::now() - began > std::chrono::milliseconds(1)) {
                const hipError_t e = hipStreamSynchronize(stream);
                if (e != hipSuccess) throw EPException("HIP", "deep_ep_cpp.cpp", __LINE__, hipGetErrorString(e));
                for (; i < count; ++i)
                    if (words[i].load(std::memory_order_acquire) == kUnset)
                        throw EPException("HIP", "deep_ep_cpp.cpp", __LINE__, "the kernel did not report its end");
            }
        }
        return words[count - 1].load(std::memory_order_acquire);
    }
};

// reference: csrc/kernels/efa_kernels.cu:1591-1651 (the host wait for the total is the reference's .item())
static std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, int64_t, torch::Tensor> routing_sort_impl(
    const torch::Tensor& is_token_in_rank, bool with_positions) {
    EP_HOST_ASSERT(is_token_in_rank.dim() == 2);
    EP_HOST_ASSERT(is_token_in_rank.scalar_type() == torch::kBool);
    EP_HOST_ASSERT(is_token_in_rank.is_contiguous());
    EP_HOST_ASSERT(is_token_in_rank.is_cuda());
    // the total is waited for, which a stream that is being captured cannot give
    EP_HOST_ASSERT(c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None);
    const int num_tokens = static_cast<int>(is_token_in_rank.size(0)), num_ranks = static_cast<int>(is_token_in_rank.size(1));
    const int64_t pairs = int64_t(num_tokens) * num_ranks;
    const int64_t ws_bytes = std::max<int64_t>(256, int64_t(deepep_routing_sort_workspace_bytes(num_tokens, num_ranks)));
    ResultBlock b;
    const int64_t counts_at = b.reserve(4 * num_ranks), cumsum_at = b.reserve(8 * (num_ranks + 1)), ws_at = b.reserve(ws_bytes);
    const int64_t ids_at = b.reserve(8 * std::max<int64_t>(1, pairs)), positions_at = b.reserve(with_positions ? 4 * pairs : 0);
    b.allocate(is_token_in_rank.device());
    auto send_counts = b.take(counts_at, {num_ranks}, torch::kInt32);
    auto send_cumsum = b.take(cumsum_at, {num_ranks + 1}, torch::kInt64);
    torch::Tensor row_of_pair;
    if (with_positions) row_of_pair = b.take(positions_at, {num_tokens, num_ranks}, torch::kInt32);
    uint8_t* base = b.block.data_ptr<uint8_t>();
    const auto* member = reinterpret_cast<const uint8_t*>(is_token_in_rank.data_ptr<bool>());
    const HostWords report(deepep_routing_sort_report_words(member, num_tokens, num_ranks));
    const hipStream_t stream = current_stream();
    abi_check(deepep_moe_routing_sort_reporting(
        member, num_tokens, num_ranks,
        reinterpret_cast<int64_t*>(base + ids_at), send_counts.data_ptr<int>(), send_cumsum.data_ptr<int64_t>(),
        with_positions and num_tokens > 0 ? row_of_pair.data_ptr<int>() : nullptr, report.device_pointer(),
        base + ws_at, size_t(ws_bytes), stream));
    const int64_t total = report.wait(stream);
    return {b.take(ids_at, {total}, torch::kInt64), send_counts, send_cumsum, total, row_of_pair};
}

static std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, int64_t> moe_routing_sort(const torch::Tensor& is_token_in_rank) {
    auto [ids, counts, cumsum, total, unused] = routing_sort_impl(is_token_in_rank, false);
    (void)unused;
    return {ids, counts, cumsum, total};
}

// The same plus row_of_pair [T, R] int32, the inverse of the list, which combine_reduce takes to run as one launch.
static std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, int64_t, torch::Tensor> moe_routing_sort_with_positions(
    const torch::Tensor& is_token_in_rank) {
    return routing_sort_impl(is_token_in_rank, true);
}

// reference: csrc/kernels/intranode.cu:90-112 (the channel part of notify_dispatch)
static torch::Tensor channel_prefix_matrix(const torch::Tensor& is_token_in_rank, int num_channels) {
    EP_HOST_ASSERT(is_token_in_rank.dim() == 2 and is_token_in_rank.is_contiguous() and is_token_in_rank.is_cuda());
    EP_HOST_ASSERT(is_token_in_rank.scalar_type() == torch::kBool);
    EP_HOST_ASSERT(num_channels > 0);
    const int num_tokens = static_cast<int>(is_token_in_rank.size(0)), num_ranks = static_cast<int>(is_token_in_rank.size(1));
    auto cpm = empty_on(is_token_in_rank.device(), {num_ranks, num_channels}, torch::kInt32);
    abi_check(deepep_channel_prefix_matrix(reinterpret_cast<const uint8_t*>(is_token_in_rank.data_ptr<bool>()),
                                           num_tokens, num_ranks, num_channels, cpm.data_ptr<int>(), current_stream()));
    return cpm;
}

// reference: csrc/kernels/efa_kernels.cu:1653-1691 (same arguments, same outputs)
static std::tuple<torch::Tensor, torch::Tensor> topk_remap(const torch::Tensor& topk_idx, const torch::Tensor& topk_weights,
                                                           const torch::Tensor& sorted_token_ids,
                                                           const torch::Tensor& send_cumsum, int64_t total_send,
                                                           int num_ranks, int num_local_experts) {
    EP_HOST_ASSERT(topk_idx.dim() == 2);
    EP_HOST_ASSERT(topk_idx.is_contiguous() && topk_idx.is_cuda());
    EP_HOST_ASSERT(topk_weights.dim() == 2);
    EP_HOST_ASSERT(topk_weights.is_contiguous() && topk_weights.is_cuda());
    EP_HOST_ASSERT(topk_idx.scalar_type() == torch::kInt64 and topk_weights.scalar_type() == torch::kFloat32);
    EP_HOST_ASSERT(topk_weights.size(0) == topk_idx.size(0) and topk_weights.size(1) == topk_idx.size(1));
    EP_HOST_ASSERT(sorted_token_ids.scalar_type() == torch::kInt64 and sorted_token_ids.is_contiguous());
    EP_HOST_ASSERT(send_cumsum.scalar_type() == torch::kInt64 and send_cumsum.is_contiguous());
    EP_HOST_ASSERT(send_cumsum.numel() == num_ranks + 1);
    EP_HOST_ASSERT(total_send >= 0 and total_send <= sorted_token_ids.numel());
    const int num_topk = static_cast<int>(topk_idx.size(1));
    ResultBlock b;
    const int64_t topk_at = b.reserve(8 * total_send * num_topk), weights_at = b.reserve(4 * total_send * num_topk);
    b.allocate(topk_idx.device());
    auto remapped_topk = b.take(topk_at, {total_send, num_topk}, torch::kInt64);
    auto remapped_weights = b.take(weights_at, {total_send, num_topk}, torch::kFloat32);
    abi_check(deepep_topk_remap(topk_idx.data_ptr<int64_t>(), topk_weights.data_ptr<float>(),
                                sorted_token_ids.data_ptr<int64_t>(), send_cumsum.data_ptr<int64_t>(),
                                static_cast<int>(topk_idx.size(0)), num_topk, num_ranks, num_local_experts, total_send,
                                remapped_topk.data_ptr<int64_t>(), remapped_weights.data_ptr<float>(), current_stream()));
    return {remapped_topk, remapped_weights};
}

// reference: csrc/kernels/efa_kernels.cu:1726-1749 (recv_counts is accepted and not needed: the prefix has it)
static torch::Tensor build_recv_src_meta(const torch::Tensor& recv_counts, const torch::Tensor& recv_cumsum,
                                         int64_t num_recv_tokens, int num_ranks, int num_local_ranks) {
    EP_HOST_ASSERT(recv_counts.is_cuda() and recv_cumsum.is_cuda());
    EP_HOST_ASSERT(recv_cumsum.scalar_type() == torch::kInt64 and recv_cumsum.is_contiguous());
    EP_HOST_ASSERT(recv_cumsum.numel() == num_ranks + 1 and num_recv_tokens >= 0);
    auto meta = empty_on(recv_cumsum.device(), {num_recv_tokens, 8}, torch::kUInt8);
    abi_check(deepep_build_recv_src_meta(recv_cumsum.data_ptr<int64_t>(), num_ranks, num_local_ranks, num_recv_tokens,
                                         meta.data_ptr<uint8_t>(), current_stream()));
    return meta;
}

// ---------------------------------------------------------------------------
// The calls of ll_runtime.AllToAllState.  A call is given the state and takes the tensors out of its attribute
// dictionary by interned name, or asks the state where a subclass keeps one elsewhere (a property), so whatever the
// attributes hold at that moment is what the kernels get; through ctypes the argument lists cost the host 5 us a call
// on top of the launch, and the ten results of the metadata call 14 us more.
// ---------------------------------------------------------------------------
struct Attributes {
    PyObject* object;                            // null: a plain dictionary
    pybind11::object dict;
    mutable std::vector<pybind11::object> held;  // what came from elsewhere

    explicit Attributes(const pybind11::handle& v) {
        object = PyDict_Check(v.ptr()) ? nullptr : v.ptr();
        dict = object == nullptr ? pybind11::reinterpret_borrow<pybind11::object>(v)
                                 : pybind11::reinterpret_steal<pybind11::object>(PyObject_GenericGetDict(object, nullptr));
        if (!dict) PyErr_Clear();
    }
    PyObject* get(PyObject* key) const {
        PyObject* v = dict ? PyDict_GetItemWithError(dict.ptr(), key) : nullptr;  // borrowed
        if (v == nullptr) {
            if (PyErr_Occurred()) throw pybind11::error_already_set();
            if (object == nullptr) {
                PyErr_SetObject(PyExc_AttributeError, key);
                throw pybind11::error_already_set();
            }
            v = PyObject_GetAttr(object, key);
            if (v == nullptr) throw pybind11::error_already_set();
            held.push_back(pybind11::reinterpret_steal<pybind11::object>(v));
        }
        return v;
    }
    const torch::Tensor* tensor(PyObject* key) const {
        PyObject* v = get(key);
        if (v == Py_None) return nullptr;
        if (!THPVariable_Check(v)) throw pybind11::type_error("a tensor or None was expected");
        return &THPVariable_Unpack(v);
    }
    template <typename T = void>
    T* ptr(PyObject* key) const {
        const torch::Tensor* t = tensor(key);
        return t != nullptr ? static_cast<T*>(t->data_ptr()) : nullptr;
    }
    int64_t size_bytes(PyObject* key) const {
        const torch::Tensor* t = tensor(key);
        return t != nullptr ? int64_t(t->nbytes()) : 0;
    }
    int64_t integer(PyObject* key) const {
        const int64_t v = PyLong_AsLongLong(get(key));
        if (v == -1 and PyErr_Occurred()) throw pybind11::error_already_set();
        return v;
    }
};

// An attribute name as the interned string Python's own lookups use; made once, when the module is loaded.
#define DEEPEP_NAME(x) static PyObject* const x = PyUnicode_InternFromString(#x)

template <typename T = void>
static T* optional_ptr(const std::optional<torch::Tensor>& t) {
    return t.has_value() ? static_cast<T*>(t->data_ptr()) : nullptr;
}

// A failed call raises what the ctypes view of the library raises.
static void capi_check(int rc) {
    if (rc == 0) return;
    const pybind11::object kind = pybind11::module_::import("deepep_efa_amd._capi").attr("DeepEPError");
    PyErr_SetString(kind.ptr(), deepep_last_error());
    throw pybind11::error_already_set();
}

// f(args...) with the GIL released, as the ctypes view calls the library: a launch that waits for a full queue does
// not hold up the other Python threads.
template <typename... P, typename... A>
static int without_gil(int (*f)(P...), A... args) {
    const pybind11::gil_scoped_release release;
    return f(args...);
}
template <typename... P, typename... A>
static void capi_call(int (*f)(P...), A... args) {
    capi_check(without_gil(f, args...));
}

// reference: csrc/transport/ll_pipeline.cpp:1204-1269,1277-1361 — the bookkeeping between the gather of the
// route counts and the exchange, on the stream instead of on the host.
struct ExchangeMetadata {
    torch::Tensor send_counts, recv_counts, totals, combine_remote_recv_offset, num_recv_tokens, tokens_per_expert;
    ResultBlock block;
    int64_t records_at, record_pitch, capacity;  // source_rank / source_offset / padded_index / combine_send_offset

    torch::Tensor record(int i) const { return block.take(records_at + i * record_pitch, {capacity}, torch::kInt32); }
};

// The launch's return code is left to the caller, whose callers know different exceptions for it.
static int exchange_metadata_of(const torch::Tensor& all_num_routed, int rank, int max_tokens, int64_t row_capacity,
                                int64_t record_pitch, ExchangeMetadata& m) {
    const int num_ranks = static_cast<int>(all_num_routed.size(0)), num_experts = static_cast<int>(all_num_routed.size(1));
    const int64_t r = num_ranks, el = num_experts / std::max(num_ranks, 1);
    m.capacity = std::max<int64_t>(row_capacity, 0), m.record_pitch = record_pitch;
    ResultBlock& b = m.block;
    const int64_t send_at = b.reserve(4 * r), recv_at = b.reserve(4 * r), totals_at = b.reserve(12);
    const int64_t remote_at = b.reserve(8 * r), num_at = b.reserve(8), per_expert_at = b.reserve(4 * el);
    m.records_at = b.reserve(4 * record_pitch);
    b.allocate(all_num_routed.device());
    const auto i32 = torch::kInt32;
    m.send_counts = b.take(send_at, {r}, i32), m.recv_counts = b.take(recv_at, {r}, i32);
    m.totals = b.take(totals_at, {3}, i32), m.combine_remote_recv_offset = b.take(remote_at, {r}, torch::kInt64);
    m.num_recv_tokens = b.take(num_at, {2}, i32), m.tokens_per_expert = b.take(per_expert_at, {el}, i32);
    auto at = [&](int64_t offset) { return static_cast<uint8_t*>(b.block.data_ptr()) + offset; };
    auto record = [&](int i) { return reinterpret_cast<uint32_t*>(at(m.records_at + i * record_pitch)); };
    return without_gil(&deepep_ll_exchange_metadata, static_cast<const int32_t*>(all_num_routed.data_ptr()), num_experts,
                       num_ranks, rank, max_tokens, row_capacity, reinterpret_cast<int32_t*>(at(send_at)),
                       reinterpret_cast<int32_t*>(at(recv_at)), reinterpret_cast<int32_t*>(at(totals_at)),
                       reinterpret_cast<int64_t*>(at(remote_at)), record(0), record(1), record(2), record(3),
                       reinterpret_cast<uint32_t*>(at(num_at)), reinterpret_cast<uint32_t*>(at(per_expert_at)),
                       current_stream());
}

// Returns (send_counts [R] i32, recv_counts [R] i32, totals [3] i32 = sent / received / corrupt,
// combine_remote_recv_offset [R] i64, records [4, row_capacity] i32 = source_rank / source_offset / padded_index /
// combine_send_offset, num_recv_tokens [2] i32, tokens_per_expert [E_l] i32).
static std::tuple<torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor>
ll_exchange_metadata(const torch::Tensor& all_num_routed, int rank, int num_max_dispatch_tokens_per_rank,
                     int64_t row_capacity) {
    EP_HOST_ASSERT(all_num_routed.dim() == 2 and all_num_routed.is_contiguous() and all_num_routed.is_cuda());
    EP_HOST_ASSERT(all_num_routed.scalar_type() == torch::kInt32);
    EP_HOST_ASSERT(row_capacity >= 0);
    EP_HOST_ASSERT(all_num_routed.size(0) > 0 and all_num_routed.size(1) % all_num_routed.size(0) == 0);
    ExchangeMetadata m;
    abi_check(exchange_metadata_of(all_num_routed, rank, num_max_dispatch_tokens_per_rank, row_capacity, 4 * row_capacity, m));
    return {m.send_counts, m.recv_counts, m.totals, m.combine_remote_recv_offset,
            m.block.take(m.records_at, {4, row_capacity}, torch::kInt32), m.num_recv_tokens, m.tokens_per_expert};
}

namespace name {
DEEPEP_NAME(send_counts);
DEEPEP_NAME(recv_counts);
DEEPEP_NAME(totals);
DEEPEP_NAME(combine_remote_recv_offset);
DEEPEP_NAME(source_rank);
DEEPEP_NAME(source_offset);
DEEPEP_NAME(padded_index);
DEEPEP_NAME(combine_send_offset);
DEEPEP_NAME(num_recv_tokens);
DEEPEP_NAME(tokens_per_expert);
DEEPEP_NAME(send_rows);
DEEPEP_NAME(send_capacity);
DEEPEP_NAME(send_count);
DEEPEP_NAME(send_expert_prefix);
DEEPEP_NAME(send_cumsum);
DEEPEP_NAME(pair_slot);
DEEPEP_NAME(workspace);
DEEPEP_NAME(slot_rows);
DEEPEP_NAME(row_capacity);
DEEPEP_NAME(recv_by_source);
DEEPEP_NAME(by_source_workspace);
DEEPEP_NAME(record_packed_row);
DEEPEP_NAME(packed_recv_x);
DEEPEP_NAME(packed_recv_scales);
DEEPEP_NAME(packed_recv_count);
DEEPEP_NAME(packed_recv_src_info);
DEEPEP_NAME(packed_recv_layout_range);
DEEPEP_NAME(send_flat);
DEEPEP_NAME(recv_flat);
DEEPEP_NAME(expected_rows);
}  // namespace name

// The same by name, every record an array of its own.
static pybind11::dict exchange_metadata_dict(const torch::Tensor& all_num_routed, int rank, int max_tokens,
                                             int64_t capacity) {
    using namespace name;
    if (all_num_routed.dim() != 2) throw pybind11::value_error("the route counts are [ranks, experts]");
    ExchangeMetadata m;
    const int64_t pitch = align_up<int64_t>(4 * std::max<int64_t>(capacity, 0), 256);
    capi_check(exchange_metadata_of(all_num_routed, rank, max_tokens, capacity, pitch, m));
    pybind11::dict out;
    auto put = [&](PyObject* key, const torch::Tensor& t) {
        PyObject* v = THPVariable_Wrap(t);
        const bool ok = v != nullptr and PyDict_SetItem(out.ptr(), key, v) == 0;
        Py_XDECREF(v);
        if (!ok) throw pybind11::error_already_set();
    };
    put(send_counts, m.send_counts), put(recv_counts, m.recv_counts), put(totals, m.totals);
    put(combine_remote_recv_offset, m.combine_remote_recv_offset);
    put(source_rank, m.record(0)), put(source_offset, m.record(1)), put(padded_index, m.record(2));
    put(combine_send_offset, m.record(3)), put(num_recv_tokens, m.num_recv_tokens);
    put(tokens_per_expert, m.tokens_per_expert);
    return out;
}

struct AllToAllCalls {
    int num_ranks, rank, num_experts, max_tokens, hidden, num_topk, fmt;

    void dispatch_send(const pybind11::handle& state, const torch::Tensor& x, const torch::Tensor& topk_idx) const {
        using namespace name;
        const Attributes s(state);
        capi_call(
            &deepep_ll_dispatch_send_by_dest,
            x.data_ptr(), static_cast<const int64_t*>(topk_idx.data_ptr()), static_cast<int>(x.size(0)), hidden,
            num_topk, num_experts, num_ranks, rank, max_tokens, fmt, s.ptr(send_rows), s.integer(send_capacity),
            s.ptr<int32_t>(send_count), s.ptr<int32_t>(send_expert_prefix), s.ptr<int32_t>(send_counts),
            s.ptr<int64_t>(send_cumsum), s.ptr<int32_t>(pair_slot), s.ptr(workspace), size_t(s.size_bytes(workspace)),
            current_stream());
    }

    void dispatch_recv_ordered(const pybind11::handle& state, const torch::Tensor& all_num_routed,
                               const std::optional<torch::Tensor>& stats) const {
        using namespace name;
        const Attributes s(state);
        capi_call(
            &deepep_ll_dispatch_recv_by_source_ordered,
            s.ptr(recv_by_source), s.integer(slot_rows), static_cast<const int32_t*>(all_num_routed.data_ptr()), hidden,
            num_experts, num_ranks, rank, max_tokens, fmt, s.ptr(packed_recv_x), s.ptr(packed_recv_scales),
            s.ptr<int32_t>(packed_recv_src_info), s.ptr<int64_t>(packed_recv_layout_range),
            s.ptr<int32_t>(packed_recv_count), optional_ptr<int32_t>(stats), s.ptr<uint32_t>(tokens_per_expert),
            s.ptr<int32_t>(record_packed_row), s.integer(row_capacity), s.integer(expected_rows),
            s.ptr(by_source_workspace), size_t(s.size_bytes(by_source_workspace)), current_stream());
    }

    void dispatch_recv(const pybind11::handle& state, const pybind11::dict& meta,
                       const std::optional<torch::Tensor>& stats) const {
        using namespace name;
        const Attributes s(state), m(meta);
        capi_call(
            &deepep_ll_dispatch_recv_by_source,
            s.ptr(recv_by_source), s.integer(slot_rows), m.ptr<int32_t>(recv_counts), m.ptr<uint32_t>(source_offset),
            m.ptr<uint32_t>(num_recv_tokens), s.integer(row_capacity), hidden, num_experts, num_ranks, max_tokens, fmt,
            s.ptr(packed_recv_x), s.ptr(packed_recv_scales), s.ptr<int32_t>(packed_recv_src_info),
            s.ptr<int64_t>(packed_recv_layout_range), s.ptr<int32_t>(packed_recv_count), optional_ptr<int32_t>(stats),
            s.ptr<uint32_t>(tokens_per_expert), s.ptr<int32_t>(record_packed_row), s.integer(expected_rows),
            s.ptr(by_source_workspace), size_t(s.size_bytes(by_source_workspace)), current_stream());
    }

    void combine_send(const pybind11::handle& state, const pybind11::dict& meta, const torch::Tensor& y,
                      const std::optional<torch::Tensor>& peer_recv_flat,
                      const std::optional<torch::Tensor>& peer_recv_rows) const {
        using namespace name;
        const Attributes s(state), m(meta);
        capi_call(
            &deepep_ll_combine_send_by_dest,
            y.data_ptr(), s.ptr<int32_t>(record_packed_row), m.ptr<uint32_t>(source_rank),
            m.ptr<uint32_t>(padded_index), m.ptr<uint32_t>(combine_send_offset), m.ptr<uint32_t>(num_recv_tokens),
            s.integer(row_capacity), hidden, num_experts, num_ranks, max_tokens, s.ptr(send_flat),
            m.ptr<int32_t>(recv_counts), m.ptr<int64_t>(combine_remote_recv_offset),
            optional_ptr<void*>(peer_recv_flat), optional_ptr<int64_t>(peer_recv_rows), s.integer(expected_rows),
            current_stream());
    }

    void combine_recv(const pybind11::handle& state, const torch::Tensor& topk_idx, const torch::Tensor& topk_weights,
                      const torch::Tensor& out, const std::optional<torch::Tensor>& recv, int64_t recv_slot_rows,
                      bool accumulate) const {
        using namespace name;
        const Attributes s(state);
        const torch::Tensor* buf = recv.has_value() ? &recv.value() : s.tensor(recv_flat);
        if (buf == nullptr) throw pybind11::type_error("recv is None and so is recv_flat");
        capi_call(
            &deepep_ll_combine_recv_flat,
            buf->data_ptr(), buf->size(0), recv_slot_rows, s.ptr<int32_t>(send_expert_prefix),
            static_cast<const int64_t*>(topk_idx.data_ptr()), static_cast<const float*>(topk_weights.data_ptr()),
            s.ptr<int32_t>(pair_slot), static_cast<int>(topk_idx.size(0)), hidden, num_topk, num_experts, num_ranks,
            max_tokens, accumulate ? 1 : 0, out.data_ptr(), current_stream());
    }
};

// reference: deep_ep/buffer.py:1542-1557 — zero_() + index_add_ over the returned rows, then the biases
static std::tuple<torch::Tensor, std::optional<torch::Tensor>> combine_reduce(
    const torch::Tensor& recv_x, const std::optional<torch::Tensor>& recv_topk_weights,
    const torch::Tensor& sorted_token_ids, const torch::Tensor& send_cumsum, const torch::Tensor& is_token_in_rank,
    const std::optional<torch::Tensor>& bias_0, const std::optional<torch::Tensor>& bias_1,
    const std::optional<torch::Tensor>& row_of_pair) {
    EP_HOST_ASSERT(recv_x.dim() == 2 and recv_x.is_contiguous() and recv_x.is_cuda());
    EP_HOST_ASSERT(recv_x.scalar_type() == torch::kBFloat16);
    EP_HOST_ASSERT(is_token_in_rank.dim() == 2 and is_token_in_rank.is_contiguous());
    EP_HOST_ASSERT(is_token_in_rank.scalar_type() == torch::kBool);
    EP_HOST_ASSERT(sorted_token_ids.scalar_type() == torch::kInt64 and sorted_token_ids.is_contiguous());
    EP_HOST_ASSERT(send_cumsum.scalar_type() == torch::kInt64 and send_cumsum.is_contiguous());
    const int num_tokens = static_cast<int>(is_token_in_rank.size(0)), num_ranks = static_cast<int>(is_token_in_rank.size(1));
    const int hidden = static_cast<int>(recv_x.size(1));
    EP_HOST_ASSERT(send_cumsum.numel() == num_ranks + 1);
    const int64_t max_rows = std::min<int64_t>(recv_x.size(0), sorted_token_ids.numel());
    int num_topk = 0;
    if (recv_topk_weights.has_value()) {
        EP_HOST_ASSERT(recv_topk_weights->dim() == 2 and recv_topk_weights->is_contiguous());
        EP_HOST_ASSERT(recv_topk_weights->scalar_type() == torch::kFloat32 and recv_topk_weights->size(0) >= max_rows);
        num_topk = static_cast<int>(recv_topk_weights->size(1));
    }
    for (const auto* b : {&bias_0, &bias_1})
        if (b->has_value()) {
            EP_HOST_ASSERT((*b)->dim() == 2 and (*b)->is_contiguous() and (*b)->scalar_type() == torch::kBFloat16);
            EP_HOST_ASSERT((*b)->size(0) == num_tokens and (*b)->size(1) == hidden);
        }
    if (row_of_pair.has_value()) {
        EP_HOST_ASSERT(row_of_pair->scalar_type() == torch::kInt32 and row_of_pair->is_contiguous() and row_of_pair->is_cuda());
        EP_HOST_ASSERT(row_of_pair->dim() == 2 and row_of_pair->size(0) == num_tokens and row_of_pair->size(1) == num_ranks);
    }
    auto combined_x = empty_on(recv_x.device(), {num_tokens, hidden}, torch::kBFloat16);
    std::optional<torch::Tensor> combined_w;
    if (recv_topk_weights.has_value())
        combined_w = empty_on(recv_topk_weights->device(), {num_tokens, num_topk}, torch::kFloat32);
    torch::Tensor ws;  // where the pairs' rows are looked up, unless the sort's table is given
    if (!row_of_pair.has_value())
        ws = empty_on(recv_x.device(),
                      {std::max<int64_t>(256, int64_t(deepep_combine_reduce_workspace_bytes(num_tokens, num_ranks)))},
                      torch::kUInt8);
    abi_check(deepep_combine_reduce(
        recv_x.data_ptr(), recv_topk_weights.has_value() ? recv_topk_weights->data_ptr<float>() : nullptr,
        sorted_token_ids.data_ptr<int64_t>(), send_cumsum.data_ptr<int64_t>(),
        reinterpret_cast<const uint8_t*>(is_token_in_rank.data_ptr<bool>()),
        bias_0.has_value() ? bias_0->data_ptr() : nullptr, bias_1.has_value() ? bias_1->data_ptr() : nullptr, num_tokens,
        hidden, num_topk, num_ranks, max_rows, row_of_pair.has_value() ? row_of_pair->data_ptr<int>() : nullptr,
        combined_x.data_ptr(),
        combined_w.has_value() ? combined_w->data_ptr<float>() : nullptr,
        ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? size_t(ws.numel()) : 0,
        current_stream()));
    return {combined_x, combined_w};
}

// reference: deep_ep/buffer.py:877,917 — send_x = x[sorted_ids], send_scales = scales[sorted_ids]
static std::tuple<torch::Tensor, std::optional<torch::Tensor>> pack_rows(const torch::Tensor& x,
                                                                         const std::optional<torch::Tensor>& x_scales,
                                                                         const torch::Tensor& sorted_token_ids,
                                                                         const torch::Tensor& send_cumsum) {
    EP_HOST_ASSERT(x.dim() == 2 and x.is_contiguous() and x.is_cuda());
    EP_HOST_ASSERT(sorted_token_ids.dim() == 1 and sorted_token_ids.is_contiguous());
    EP_HOST_ASSERT(sorted_token_ids.scalar_type() == torch::kInt64);
    EP_HOST_ASSERT(send_cumsum.scalar_type() == torch::kInt64 and send_cumsum.is_contiguous() and send_cumsum.numel() >= 1);
    const int64_t rows = sorted_token_ids.numel();
    const int64_t row_bytes = x.size(1) * x.element_size();
    EP_HOST_ASSERT(row_bytes % 16 == 0);
    auto out = empty_on(x.device(), {rows, x.size(1)}, x.scalar_type());
    std::optional<torch::Tensor> out_scales;
    int64_t scale_row_bytes = 0;
    if (x_scales.has_value()) {
        EP_HOST_ASSERT(x_scales->dim() == 2 and x_scales->is_contiguous() and x_scales->size(0) == x.size(0));
        scale_row_bytes = x_scales->size(1) * x_scales->element_size();
        EP_HOST_ASSERT(scale_row_bytes % 4 == 0);
        out_scales = empty_on(x_scales->device(), {rows, x_scales->size(1)}, x_scales->scalar_type());
    }
    const int num_ranks = static_cast<int>(send_cumsum.numel() - 1);
    const int64_t* cumsum = send_cumsum.data_ptr<int64_t>();
    abi_check(deepep_pack_rows_by_rank(
        x.data_ptr(), x_scales.has_value() ? x_scales->data_ptr() : nullptr, sorted_token_ids.data_ptr<int64_t>(),
        cumsum + num_ranks, num_ranks > 0 ? cumsum : nullptr, num_ranks, rows, static_cast<int>(x.size(0)),
        static_cast<int>(row_bytes), static_cast<int>(scale_row_bytes), out.data_ptr(),
        out_scales.has_value() ? out_scales->data_ptr() : nullptr, current_stream()));
    return {out, out_scales};
}

// ---------------------------------------------------------------------------
// The calls a step makes as plain C functions (METH_FASTCALL) for the Python methods around them: arguments by
// position, converted one by one.  pybind11's dispatcher takes 0.3 to 0.5 us of host time a call more, of the 4 to 5
// that a call with its launch takes, and small steps are bound by that.
// ---------------------------------------------------------------------------
static const torch::Tensor& tensor_argument(PyObject* v) {
    if (!THPVariable_Check(v)) throw pybind11::type_error("a torch.Tensor was expected");
    return THPVariable_Unpack(v);
}
static const torch::Tensor* optional_tensor_argument(PyObject* v) { return v == Py_None ? nullptr : &tensor_argument(v); }
// Numbers and truth values by pybind11's own rules, implicit conversions included: what it refuses for a bound
// function (a float for an int, a str or a list for a bool) is refused here, with the same TypeError.
template <typename T>
static T scalar_argument(PyObject* v) {
    pybind11::detail::make_caster<T> caster;
    if (!caster.load(v, true)) throw pybind11::type_error("incompatible function arguments");
    return pybind11::detail::cast_op<T>(caster);
}
template <typename T>
static T& object_argument(PyObject* v) {
    pybind11::detail::make_caster<T> caster;
    if (!caster.load(v, true) or v == Py_None) throw pybind11::type_error("incompatible function arguments");
    return pybind11::detail::cast_op<T&>(caster);
}
static int int_argument(PyObject* v) { return scalar_argument<int>(v); }
static bool bool_argument(PyObject* v) { return scalar_argument<bool>(v); }

template <typename A>
struct Argument;
template <>
struct Argument<const torch::Tensor&> {
    const torch::Tensor& value;
    explicit Argument(PyObject* v) : value(tensor_argument(v)) {}
};
template <>
struct Argument<const std::optional<torch::Tensor>&> {
    std::optional<torch::Tensor> value;
    explicit Argument(PyObject* v) {
        if (v != Py_None) value = tensor_argument(v);
    }
};
template <>
struct Argument<std::optional<EventHandle>&> {
    std::optional<EventHandle> value;
    explicit Argument(PyObject* v) {
        if (v != Py_None) value = object_argument<EventHandle>(v);
    }
};
template <>
struct Argument<const pybind11::handle&> {
    pybind11::handle value;
    explicit Argument(PyObject* v) : value(v) {}
};
template <>
struct Argument<const pybind11::dict&> {
    pybind11::dict value;
    explicit Argument(PyObject* v) : value(pybind11::reinterpret_borrow<pybind11::dict>(v)) {
        if (!PyDict_Check(v)) throw pybind11::type_error("a dict was expected");
    }
};
template <>
struct Argument<int> {
    int value;
    explicit Argument(PyObject* v) : value(int_argument(v)) {}
};
template <>
struct Argument<int64_t> {
    int64_t value;
    explicit Argument(PyObject* v) : value(scalar_argument<int64_t>(v)) {}
};
template <>
struct Argument<bool> {
    bool value;
    explicit Argument(PyObject* v) : value(bool_argument(v)) {}
};

static pybind11::object result_object(const torch::Tensor& t) {
    PyObject* v = THPVariable_Wrap(t);  // None for an undefined one
    if (v == nullptr) throw pybind11::error_already_set();
    return pybind11::reinterpret_steal<pybind11::object>(v);
}
static pybind11::object result_object(int64_t n) { return pybind11::int_(n); }
static pybind11::object result_object(const EventHandle& e) { return pybind11::cast(e); }
static pybind11::object result_object(const pybind11::dict& d) { return d; }
template <typename T>
static pybind11::object result_object(const std::optional<T>& v) {
    if (!v.has_value()) return pybind11::none();
    return result_object(*v);
}
template <typename... T>
static pybind11::object result_object(const std::tuple<T...>& v) {
    return std::apply(
        [](const T&... item) {
            pybind11::tuple out(sizeof...(T));
            Py_ssize_t i = 0;
            (PyTuple_SET_ITEM(out.ptr(), i++, result_object(item).release().ptr()), ...);
            return pybind11::object(std::move(out));
        },
        v);
}

// Runs f and turns what it throws into the Python error that pybind11 raises for a bound function: its registered
// translators, PyTorch's among them (torch.OutOfMemoryError, torch.AcceleratorError), have their say.
template <typename F>
static PyObject* as_python_call(Py_ssize_t got, Py_ssize_t wanted, F&& f) {
    try {
        if (got != wanted) throw pybind11::type_error("wrong number of arguments");
        return f().release().ptr();
    } catch (pybind11::error_already_set& e) {
        e.restore();
    } catch (...) {
        pybind11::detail::try_translate_exceptions();
    }
    return nullptr;
}

// PlainCall<&f>::call is f as a METH_FASTCALL function; a member function takes its object first.
template <auto F>
struct PlainCall;

template <typename R, typename... A, R (*F)(A...)>
struct PlainCall<F> {
    template <size_t... I>
    static pybind11::object with(PyObject* const* a, std::index_sequence<I...>) {
        std::tuple<Argument<A>...> given{Argument<A>(a[I])...};
        return result_object(F(std::get<I>(given).value...));
    }
    static PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
        return as_python_call(n, sizeof...(A), [&] { return with(a, std::index_sequence_for<A...>()); });
    }
};

template <typename C, typename M, typename R, typename... A>
struct PlainMemberCall {
    template <M F, size_t... I>
    static pybind11::object with(PyObject* const* a, std::index_sequence<I...>) {
        C& self = object_argument<std::remove_const_t<C>>(a[0]);
        std::tuple<Argument<A>...> given{Argument<A>(a[1 + I])...};
        if constexpr (std::is_void_v<R>) {
            (self.*F)(std::get<I>(given).value...);
            return pybind11::none();
        } else {
            return result_object((self.*F)(std::get<I>(given).value...));
        }
    }
    template <M F>
    static PyObject* run(PyObject* const* a, Py_ssize_t n) {
        return as_python_call(n, 1 + sizeof...(A), [&] { return with<F>(a, std::index_sequence_for<A...>()); });
    }
};
template <typename C, typename R, typename... A, R (C::*F)(A...)>
struct PlainCall<F> {
    static PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
        return PlainMemberCall<C, R (C::*)(A...), R, A...>::template run<F>(a, n);
    }
};
template <typename C, typename R, typename... A, R (C::*F)(A...) const>
struct PlainCall<F> {
    static PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
        return PlainMemberCall<const C, R (C::*)(A...) const, R, A...>::template run<F>(a, n);
    }
};

// The event of a low-latency call, with or without async_finish.  It is recorded before the call returns: recorded
// when somebody waits, it would also cover what the caller's stream was given in between, which takes away the
// overlap with it and hangs where that work waits for the waiter.  A record takes the stream 3 us beside kernels of
// 8 us, 1 without the fence, and the host 2; a step records two.  A dispatch's is without: what follows it are the experts,
// on a stream of this device (another's brings the fence when it waits: event.hpp).  A combine's has the fence, which a wait
// for its stream then need not bring.  Microseconds of a step, fences on both / on the combine's / on none, in a row and each waited for:
//   1 token     13.5 / 11.8 / 10.3    22.3 / 20.8 / 23.8        128   23.0 / 20.9 / 18.9    32.0 / 30.3 / 33.4
//   77 in bf16  17.4 / 15.5 / 13.7    26.2 / 24.5 / 27.5        509   25.3 / 24.0 / 22.0    33.9 / 33.0 / 35.3
static pybind11::object recorded_event(DeviceEvent::Scope scope) {
    return pybind11::cast(EventHandle(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(), scope));
}

static pybind11::object hook_object(bool wanted) {
    if (!wanted) return pybind11::none();
    return pybind11::cpp_function([] {});
}

// (buffer, x, topk_idx, stats, wait stats, max tokens, experts, use_fp8, round_scale, use_ue8m0, async, hook)
//   -> (recv_x, recv_count, handle, event, hook)
static PyObject* low_latency_dispatch_call(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return as_python_call(n, 12, [&] {
        Buffer& buffer = object_argument<Buffer>(a[0]);
        const bool use_fp8 = bool_argument(a[7]);
        LowLatencyCache& c = buffer.run_low_latency_dispatch(
            tensor_argument(a[1]), tensor_argument(a[2]), optional_tensor_argument(a[3]), optional_tensor_argument(a[4]),
            int_argument(a[5]), int_argument(a[6]), use_fp8, bool_argument(a[8]), bool_argument(a[9]));
        if (!c.handle_result) {
            c.recv_result = result_object(c.packed_recv_x);
            if (use_fp8) c.recv_result = pybind11::make_tuple(c.recv_result, result_object(c.packed_recv_scales));
            c.handle_result = pybind11::make_tuple(result_object(c.packed_recv_src_info),
                                                   result_object(c.packed_recv_layout_range), c.max_tokens, c.hidden,
                                                   c.num_experts);
        }
        (void)bool_argument(a[10]);
        const pybind11::object count = result_object(c.packed_recv_count), event = recorded_event(DeviceEvent::kLocal),
                               hook = hook_object(bool_argument(a[11]));
        return pybind11::reinterpret_steal<pybind11::object>(
            PyTuple_Pack(5, c.recv_result.ptr(), count.ptr(), c.handle_result.ptr(), event.ptr(), hook.ptr()));
    });
}

// (buffer, x, topk_idx, topk_weights, handle, wait stats, zero_copy, async, hook, out, accumulate)
//   -> (combined_x, event, hook)
static PyObject* low_latency_combine_call(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return as_python_call(n, 11, [&] {
        Buffer& buffer = object_argument<Buffer>(a[0]);
        const auto h = pybind11::reinterpret_steal<pybind11::object>(
            PySequence_Fast(a[4], "the handle of a low_latency_dispatch was expected"));
        if (!h) throw pybind11::error_already_set();
        if (PySequence_Fast_GET_SIZE(h.ptr()) != 5) throw pybind11::value_error("a handle has five entries");
        auto of_handle = [&](int i) { return PySequence_Fast_GET_ITEM(h.ptr(), i); };
        const pybind11::object combined = result_object(buffer.run_low_latency_combine(
            tensor_argument(a[1]), tensor_argument(a[2]), tensor_argument(a[3]), tensor_argument(of_handle(0)),
            tensor_argument(of_handle(1)), optional_tensor_argument(a[5]), int_argument(of_handle(2)),
            int_argument(of_handle(4)), bool_argument(a[6]), optional_tensor_argument(a[9]), bool_argument(a[10])));
        (void)bool_argument(a[7]);
        const pybind11::object event = recorded_event(DeviceEvent::kSystem), hook = hook_object(bool_argument(a[8]));
        return pybind11::reinterpret_steal<pybind11::object>(PyTuple_Pack(3, combined.ptr(), event.ptr(), hook.ptr()));
    });
}

// combine_reduce by position or by name; the last three are None unless given.
static PyObject* combine_reduce_call(PyObject*, PyObject* const* a, Py_ssize_t n, PyObject* names) {
    static constexpr const char* kNames[] = {"recv_x",           "recv_topk_weights", "sorted_token_ids", "send_cumsum",
                                             "is_token_in_rank", "bias_0",            "bias_1",           "row_of_pair"};
    constexpr Py_ssize_t kArguments = 8, kRequired = 5;
    return as_python_call(std::min(n, kArguments), n, [&] {
        PyObject* given[kArguments] = {};
        std::copy(a, a + n, given);
        for (Py_ssize_t i = 0; names != nullptr and i < PyTuple_GET_SIZE(names); ++i) {
            PyObject* const name = PyTuple_GET_ITEM(names, i);
            const auto* at = std::find_if(kNames, kNames + kArguments, [&](const char* s) {
                return PyUnicode_CompareWithASCIIString(name, s) == 0;
            });
            if (at == kNames + kArguments or given[at - kNames] != nullptr)
                throw pybind11::type_error("an argument is unknown or given twice");
            given[at - kNames] = a[n + i];
        }
        for (Py_ssize_t i = 0; i < kArguments; ++i) {
            if (given[i] == nullptr and i < kRequired) throw pybind11::type_error("an argument is missing");
            if (given[i] == nullptr) given[i] = Py_None;
        }
        return PlainCall<&combine_reduce>::with(given, std::make_index_sequence<kArguments>());
    });
}

static PyMethodDef plain(const char* name, PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t), const char* doc) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, doc};
}
static PyMethodDef plain_calls[] = {
    plain("low_latency_dispatch", low_latency_dispatch_call, "Buffer.low_latency_dispatch without its wrapper"),
    plain("low_latency_combine", low_latency_combine_call, "Buffer.low_latency_combine without its wrapper"),
    plain("get_dispatch_layout", PlainCall<&Buffer::get_dispatch_layout>::call, "Buffer.get_dispatch_layout without its wrapper"),
    plain("per_token_cast_to_fp8", PlainCall<&per_token_cast_to_fp8>::call,
          "Per-token FP8 e4m3 quantisation with 128-channel groups"),
    plain("moe_routing_sort", PlainCall<&moe_routing_sort>::call, "Token ids grouped by destination rank"),
    plain("moe_routing_sort_with_positions", PlainCall<&moe_routing_sort_with_positions>::call,
          "moe_routing_sort plus row_of_pair [T, R], the inverse of the list"),
    plain("channel_prefix_matrix", PlainCall<&channel_prefix_matrix>::call,
          "Per-rank prefix of token counts over channels"),
    plain("pack_rows", PlainCall<&pack_rows>::call, "Gather rows into per-rank contiguous send buffers"),
    plain("topk_remap", PlainCall<&topk_remap>::call,
          "Top-k of the send rows in the destination rank's expert numbering"),
    plain("build_recv_src_meta", PlainCall<&build_recv_src_meta>::call, "Source-rank metadata of the received rows"),
    {"combine_reduce", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(combine_reduce_call)),
     METH_FASTCALL | METH_KEYWORDS, "Per-token sum of the rows that came back (normal-mode combine)"},
    plain("ll_exchange_metadata", PlainCall<&ll_exchange_metadata>::call,
          "Send/receive counts, combine offsets and per-row records from the gathered route counts"),
    plain("exchange_metadata_dict", PlainCall<&exchange_metadata_dict>::call, "The same by name"),
    plain("a2a_dispatch_send", PlainCall<&AllToAllCalls::dispatch_send>::call, "AllToAllState.dispatch_send"),
    plain("a2a_dispatch_recv_ordered", PlainCall<&AllToAllCalls::dispatch_recv_ordered>::call,
          "AllToAllState.dispatch_recv_ordered"),
    plain("a2a_dispatch_recv", PlainCall<&AllToAllCalls::dispatch_recv>::call, "AllToAllState.dispatch_recv"),
    plain("a2a_combine_send", PlainCall<&AllToAllCalls::combine_send>::call, "AllToAllState.combine_send"),
    plain("a2a_combine_recv", PlainCall<&AllToAllCalls::combine_recv>::call, "AllToAllState.combine_recv"),
    {nullptr, nullptr, 0, nullptr}};

static bool is_sm90_compiled() { return true; }  // FP8 paths are always built for gfx950

}  // namespace deep_ep

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "DeepEP dispatch/combine hot path for MI355X (gfx950): host module over libdeepep_hip.so";

    pybind11::register_exception<deep_ep::EPException>(m, "EPException", PyExc_RuntimeError);

    pybind11::class_<deep_ep::Config>(m, "Config")
        .def(pybind11::init<int, int, int, int, int>(), py::arg("num_sms") = 20,
             py::arg("num_max_nvl_chunked_send_tokens") = 6, py::arg("num_max_nvl_chunked_recv_tokens") = 256,
             py::arg("num_max_rdma_chunked_send_tokens") = 6, py::arg("num_max_rdma_chunked_recv_tokens") = 256)
        .def_readonly("num_sms", &deep_ep::Config::num_sms)
        .def_readonly("num_max_nvl_chunked_send_tokens", &deep_ep::Config::num_max_nvl_chunked_send_tokens)
        .def_readonly("num_max_nvl_chunked_recv_tokens", &deep_ep::Config::num_max_nvl_chunked_recv_tokens)
        .def_readonly("num_max_rdma_chunked_send_tokens", &deep_ep::Config::num_max_rdma_chunked_send_tokens)
        .def_readonly("num_max_rdma_chunked_recv_tokens", &deep_ep::Config::num_max_rdma_chunked_recv_tokens)
        .def("get_nvl_buffer_size_hint", &deep_ep::Config::get_nvl_buffer_size_hint)
        .def("get_rdma_buffer_size_hint", &deep_ep::Config::get_rdma_buffer_size_hint);
    m.def("get_low_latency_rdma_size_hint", &deep_ep::get_low_latency_rdma_size_hint);

    pybind11::class_<deep_ep::EventHandle>(m, "EventHandle")
        .def(pybind11::init<>())
        .def("current_stream_wait", &deep_ep::EventHandle::current_stream_wait);

    pybind11::class_<deep_ep::Buffer>(m, "Buffer")
        .def(pybind11::init<int, int, int64_t, int64_t, bool, bool, bool, bool>())
        .def("is_available", &deep_ep::Buffer::is_available)
        .def("get_num_rdma_ranks", &deep_ep::Buffer::get_num_rdma_ranks)
        .def("get_rdma_rank", &deep_ep::Buffer::get_rdma_rank)
        .def("get_root_rdma_rank", &deep_ep::Buffer::get_root_rdma_rank)
        .def("get_local_device_id", &deep_ep::Buffer::get_local_device_id)
        .def("get_local_ipc_handle", &deep_ep::Buffer::get_local_ipc_handle)
        .def("get_local_buffer_tensor", &deep_ep::Buffer::get_local_buffer_tensor)
        .def("get_comm_stream", &deep_ep::Buffer::get_comm_stream)
        .def("sync", &deep_ep::Buffer::sync)
        .def("destroy", &deep_ep::Buffer::destroy)
        .def("get_dispatch_layout", &deep_ep::Buffer::get_dispatch_layout)
        .def("clean_low_latency_buffer", &deep_ep::Buffer::clean_low_latency_buffer)
        .def("low_latency_dispatch", &deep_ep::Buffer::low_latency_dispatch)
        .def("low_latency_combine", &deep_ep::Buffer::low_latency_combine, py::arg("x"), py::arg("topk_idx"),
             py::arg("topk_weights"), py::arg("src_info"), py::arg("layout_range"),
             py::arg("combine_wait_recv_cost_stats"), py::arg("num_max_dispatch_tokens_per_rank"),
             py::arg("num_experts"), py::arg("use_logfmt"), py::arg("zero_copy"), py::arg("async"),
             py::arg("return_recv_hook"), py::arg("out"), py::arg("accumulate") = false)
        .def("low_latency_update_mask_buffer", &deep_ep::Buffer::low_latency_update_mask_buffer)
        .def("low_latency_query_mask_buffer", &deep_ep::Buffer::low_latency_query_mask_buffer)
        .def("low_latency_clean_mask_buffer", &deep_ep::Buffer::low_latency_clean_mask_buffer)
        .def("get_next_low_latency_combine_buffer", &deep_ep::Buffer::get_next_low_latency_combine_buffer)
        .def("loopback_set_world", &deep_ep::Buffer::loopback_set_world)
        .def("loopback_clear_world", &deep_ep::Buffer::loopback_clear_world)
        .def("loopback_synthesise", &deep_ep::Buffer::loopback_synthesise)
        .def("loopback_own_inputs", &deep_ep::Buffer::loopback_own_inputs)
        .def("loopback_world", &deep_ep::Buffer::loopback_world)
        .def("loopback_set_combine_mode", &deep_ep::Buffer::loopback_set_combine_mode);

    if (PyModule_AddFunctions(m.ptr(), deep_ep::plain_calls) != 0) throw pybind11::error_already_set();

    pybind11::class_<deep_ep::AllToAllCalls>(m, "AllToAllCalls")
        .def(pybind11::init([](int num_ranks, int rank, int num_experts, int max_tokens, int hidden, int num_topk,
                               int fmt) {
            return deep_ep::AllToAllCalls{num_ranks, rank, num_experts, max_tokens, hidden, num_topk, fmt};
        }));

    m.def("is_sm90_compiled", deep_ep::is_sm90_compiled);
    m.attr("topk_idx_t") = py::reinterpret_borrow<py::object>(
        (PyObject*)torch::getTHPDtype(c10::CppTypeToScalarType<deep_ep::topk_idx_t>::value));
}
