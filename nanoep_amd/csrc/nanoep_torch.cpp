// PyTorch-ROCm host extension for one rank's dispatch / combine.
//
// This file owns what the reference's host pipeline owns (csrc/pipeline.cu:340-489,
// csrc/dispatch_epilogue.cpp:18-75, csrc/combine_epilogue.cpp:27-64 in the reference): argument
// validation, output allocation, stream ordering between the caller's stream and the buffer's
// communication stream, and the completion event.  All device work goes through the C ABI of
// include/nanoep_hip.h.  The module exports the reference's operator surface
// (csrc/bindings.cpp:11-86) with the same positional order, so a caller written against the
// reference's backend module binds to this one unchanged.

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/Event.h>
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>
#include <torch/extension.h>

#include <array>
#include <atomic>
#include <cstdlib>
#include <deque>
#include <exception>
#include <initializer_list>
#include <limits>
#include <memory>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "nanoep_hip.h"

namespace py = pybind11;

namespace nanoep {

using Stream = c10::hip::HIPStreamMasqueradingAsCUDA;
using StreamGuard = c10::hip::HIPStreamGuardMasqueradingAsCUDA;
using OptionalStreamGuard = c10::hip::OptionalHIPStreamGuardMasqueradingAsCUDA;
using DeviceGuard = c10::hip::HIPGuardMasqueradingAsCUDA;

namespace {

constexpr int64_t kHiddenAlignment = 256;  // the reference's H % 256 == 0 contract
constexpr double kCountTimeoutSeconds = 60.0;
// Fresh expanded dispatches whose private handle tensors the runtime keeps for callers that hand
// back only the reference's seven.
constexpr size_t kRememberedHandles = 4;
// Seven-tensor handles whose private tensors were rebuilt from the handle itself and are kept for
// its later replays.
constexpr size_t kRebuiltHandles = 64;
// Rebuilding pays from this many payload bytes written per replay on (below, the token-order walk's
// loss is smaller than what the two extra launches cost a handle that is replayed once or twice).
constexpr int64_t kRebuildPayloadBytes = int64_t{48} << 20;

// One of the library's tuning switches (no environment access: the library read it once).
int tuning_switch(const char* name) {
    int value = -1;
    return nanoep_get_tuning(name, &value) == NANOEP_OK ? value : -1;
}

void check_status(int status, const char* what) {
    if (status == NANOEP_OK)
        return;
    TORCH_CHECK(false, "nanoep ", what, " failed: ", nanoep_status_string(status), " ", nanoep_last_hip_error());
}

void check_hip(hipError_t status, const char* what) {
    TORCH_CHECK(status == hipSuccess, "HIP call ", what, " failed: ", hipGetErrorString(status));
}

Stream external_stream(int64_t handle, c10::DeviceIndex device) {
    return c10::hip::getStreamFromExternalMasqueradingAsCUDA(reinterpret_cast<hipStream_t>(handle), device);
}

bool capturing(const Stream& stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    check_hip(hipStreamIsCapturing(stream.stream(), &status), "hipStreamIsCapturing");
    return status != hipStreamCaptureStatusNone;
}

// Whether something enqueued on the stream has yet to run (never asked of a stream under capture).
bool busy(const Stream& stream) {
    const hipError_t state = hipStreamQuery(stream.stream());
    if (state == hipErrorNotReady)
        (void)hipGetLastError();  // an answer, not an error of the next call that looks for one
    return state == hipErrorNotReady;
}

// A point in a stream's work: a value the stream stores into a word of signal memory when it gets there.
// Other streams wait for the word to hold at least that value, and the host can look.  Against an event
// this is what a dependency between two streams costs here: store and wait 6 us of host time against 9 to 16
// for hipEventRecord and hipStreamWaitEvent, and 5 us between the two streams' kernels against 11 to 13.
struct StreamPoint {
    uint64_t* word = nullptr;
    uint64_t value = 0;

    bool reached() const { return __atomic_load_n(word, __ATOMIC_ACQUIRE) >= value; }
};

// The words behind StreamPoints.  A word serves one store at a time and its values only grow: it is handed
// out again when the host sees its last value there, and whoever still waits for an older one finds it
// passed.  So nothing depends on which stream used a word before, and a word needs no owner.  There are as
// many as stores were ever on their way at once, at most kMostWords a device; they stay for the process.
class StreamPoints {
   public:
    static StreamPoints& of(c10::DeviceIndex device) {
        static std::array<StreamPoints, kDevices> pools;
        return pools[static_cast<size_t>(device) % kDevices];
    }

    // A point behind everything enqueued on `stream`; none when no word is free or the device has no such
    // operations (an event serves then).
    std::optional<StreamPoint> record(const Stream& stream) {
        std::optional<StreamPoint> point = next_point(stream.device_index());
        if (!point.has_value())
            return point;
        const hipError_t status = hipStreamWriteValue64(stream.stream(), point->word, point->value, 0);
        if (status != hipSuccess) {
            (void)hipGetLastError();
            __atomic_store_n(point->word, point->value, __ATOMIC_RELEASE);  // nothing will: the word is free again
            point.reset();
        }
        return point;
    }

    static void wait(const Stream& stream, const StreamPoint& point) {
        check_hip(hipStreamWaitValue64(stream.stream(), point.word, point.value, hipStreamWaitValueGte, ~uint64_t{0}), "hipStreamWaitValue64");
    }

   private:
    static constexpr size_t kDevices = 64;
    static constexpr size_t kMostWords = 64;

    std::optional<StreamPoint> next_point(c10::DeviceIndex device) {
        std::lock_guard<std::mutex> lock(mutex_);
        for (size_t tries = 0; tries < words_.size(); ++tries) {
            StreamPoint& last = words_[next_];
            next_ = (next_ + 1) % words_.size();
            if (last.reached()) {
                ++last.value;
                return last;
            }
        }
        if (supported_ < 0) {
            int answer = 0;
            supported_ = hipDeviceGetAttribute(&answer, hipDeviceAttributeCanUseStreamWaitValue, device) == hipSuccess && answer != 0;
        }
        void* memory = nullptr;
        if (supported_ == 0 || words_.size() >= kMostWords)
            return std::nullopt;
        DeviceGuard guard(device);
        if (hipExtMallocWithFlags(&memory, sizeof(uint64_t), hipMallocSignalMemory) != hipSuccess) {
            (void)hipGetLastError();
            return std::nullopt;
        }
        __atomic_store_n(static_cast<uint64_t*>(memory), uint64_t{0}, __ATOMIC_RELEASE);
        words_.push_back(StreamPoint{static_cast<uint64_t*>(memory), 1});
        return words_.back();
    }

    std::mutex mutex_;
    std::vector<StreamPoint> words_;
    size_t next_ = 0;
    int supported_ = -1;
};

// `waiter` goes on behind what `producer` holds now.
void wait_on(const Stream& waiter, const Stream& producer) {
    if (!capturing(producer) && !capturing(waiter)) {
        if (const auto point = StreamPoints::of(producer.device_index()).record(producer)) {
            StreamPoints::wait(waiter, *point);
            return;
        }
    }
    c10::Event ready(c10::DeviceType::CUDA);
    ready.record(producer.unwrap());
    waiter.unwrap().wait(ready);
}

// Tensors are made without the dispatcher (a third of its time: an allocation of torch::empty is 1.5 us of
// a call that takes six), unless torch is to fill what is left uninitialized.
torch::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dtype, const c10::Device& device) {
    const auto& context = at::globalContext();
    if (C10_UNLIKELY(context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory()))
        return torch::empty(sizes, torch::TensorOptions().dtype(dtype).device(device));
    return torch::Tensor(at::detail::empty_cuda(sizes, dtype, device, std::nullopt));
}

// A contiguous tensor over part of another one's storage, `offset` elements of its own type from the
// storage's start.  It shares the version counter, like a view: an edit of any part through torch shows in all.
torch::Tensor part_of(const torch::Tensor& base, int64_t offset, at::IntArrayRef sizes, at::ScalarType dtype) {
    auto part = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(base.storage()), base.key_set(),
                                                         c10::scalarTypeToTypeMeta(dtype));
    auto* impl = part.unsafeGetTensorImpl();
    impl->set_storage_offset(offset);
    impl->set_sizes_contiguous(sizes);
    if (!base.is_inference())
        impl->set_version_counter(base.unsafeGetTensorImpl()->version_counter());
    return part;
}

// Compute-unit budget: 0 or the device size mean the whole device (the reference's
// resolve_main_sms, csrc/pipeline.cu:20-24).
int resolve_cu_budget(int num_sms, c10::DeviceIndex device) {
    const int device_cus = at::cuda::getDeviceProperties(device)->multiProcessorCount;
    TORCH_CHECK(num_sms >= 0 && num_sms <= device_cus, "num_sms must be between 0 and the device CU count (", device_cus, ")");
    return num_sms == device_cus ? 0 : num_sms;
}

}  // namespace

// Holds what one rank needs at world_size == 1: the device, the pinned host mailbox the layout
// kernels publish N / C into, and (only if somebody asks for it) a window-sized byte tensor.
// It keeps the reference's PeerRuntime method set (csrc/bindings.cpp:59-83) so setup code written
// for the reference runs; there are no peers, so handles are opaque tags and barriers are no-ops.
//
// dispatch and combine run without the interpreter lock, so everything here that several Python
// threads can reach at once is guarded: the mailbox by `counts_mutex_` (held by a fresh dispatch
// from the enqueue of its layout until it has read the counts), the remembered handle tensors by
// `private_mutex_`, the state flags by being atomic.
class PeerRuntime {
   public:
    PeerRuntime(int rank, int world_size, int64_t num_bytes) : num_bytes_(num_bytes) {
        TORCH_CHECK(world_size == 1 && rank == 0,
                    "this build runs one rank on one GPU (world_size == 1); got rank ", rank, " of ", world_size);
        TORCH_CHECK(num_bytes >= 0, "window size must be non-negative");
        check_hip(hipGetDevice(&device_), "hipGetDevice");
        void* mailbox = nullptr;
        check_hip(hipHostMalloc(&mailbox, NANOEP_HOST_COUNT_WORDS * sizeof(int64_t), hipHostMallocMapped | hipHostMallocCoherent),
                  "hipHostMalloc");
        host_counts_ = static_cast<int64_t*>(mailbox);
        for (int i = 0; i < NANOEP_HOST_COUNT_WORDS; ++i)
            host_counts_[i] = -1;
    }

    ~PeerRuntime() {
        if (host_counts_ != nullptr)
            (void)hipHostFree(host_counts_);
        if (rebuilt_counts_ != nullptr)
            (void)hipHostFree(rebuilt_counts_);
    }

    PeerRuntime(const PeerRuntime&) = delete;
    PeerRuntime& operator=(const PeerRuntime&) = delete;

    int rank() const { return 0; }
    int world_size() const { return 1; }
    int device() const { return device_; }

    // Every operation starts here (the reference's reserve_barrier_epochs, csrc/peer.cu:171-175):
    // a closed runtime, and one whose last fresh dispatch never got its counts, serve nothing.
    void require_usable() const {
        TORCH_CHECK(!closed_.load(), "PeerRuntime is closed");
        TORCH_CHECK(!counts_failed_.load(), "A fresh dispatch on this runtime failed while waiting for its counts; the runtime is unusable");
    }

    // One fresh dispatch's use of the mailbox, from before its layout is enqueued until the host has
    // read N and C (the reference's prepare_dispatch_counts / wait_dispatch_counts /
    // fail_dispatch_counts, csrc/peer.cu:187-232).  Fresh dispatches of other threads wait their
    // turn at the constructor.  A turn that has begun and ends without `wait` having delivered the counts
    // (a timeout, a HIP error, an exception in between) leaves the runtime failed for good: a word the
    // device stores late must never answer a later call.
    class CountsTurn {
       public:
        explicit CountsTurn(PeerRuntime& runtime) : runtime_(runtime), lock_(runtime.counts_mutex_) {
            runtime_.require_usable();
            TORCH_CHECK(!runtime_.counts_pending_.load(), "A fresh dispatch is waiting for counts or has failed");
            runtime_.counts_pending_.store(true);
        }
        CountsTurn(const CountsTurn&) = delete;
        CountsTurn& operator=(const CountsTurn&) = delete;
        ~CountsTurn() {
            if (!settled_)
                runtime_.counts_failed_.store(true);
            runtime_.counts_pending_.store(false);
        }

        int64_t* mailbox() const { return runtime_.host_counts_; }

        // The layout is enqueued next: from here on the turn needs its counts.
        void begin() { settled_ = false; }

        // Nothing was enqueued that could still write the mailbox: the turn ends without a verdict.
        void abandon() { settled_ = true; }

        // Spins until the layout enqueued on `stream` has published {N, C, A, status}.  Returns
        // NANOEP_OK or NANOEP_ERR_ROUTING (the words are complete either way); anything else throws
        // and latches the failure.
        int wait(hipStream_t stream, double timeout_seconds, int64_t (&counts)[NANOEP_HOST_COUNT_WORDS]) {
            const int status = nanoep_wait_counts(mailbox(), stream, timeout_seconds, counts);
            if (status == NANOEP_OK || status == NANOEP_ERR_ROUTING) {
                settled_ = true;
                return status;
            }
            check_status(status, "wait_counts");
            return status;
        }

       private:
        PeerRuntime& runtime_;
        std::unique_lock<std::mutex> lock_;
        bool settled_ = true;
    };

    bool counts_failed() const { return counts_failed_.load(); }

    // What a fresh dispatch whose counts never arrive leaves behind, without making a GPU misbehave:
    // a turn at the mailbox that ends with no verdict.  For tests of the failure latch.
    void lose_counts_for_test() {
        CountsTurn lost(*this);
        lost.begin();
    }

    // Whether fresh dispatches should allocate their outputs after the counts are known: set when a
    // call that allocated at the upper bound turned out to hold over 1.25 times what it used (many
    // masked choices), cleared when an exact call shows that the bound would have been close enough.
    bool prefers_exact_outputs() const { return prefers_exact_outputs_.load(); }
    void note_output_fill(bool bound_was_close) { prefers_exact_outputs_.store(!bound_was_close); }

    // Rows the latest fresh dispatch of a geometry ended up using.  Where the upper bound of the output
    // shapes is not close (large alignment gaps), a fresh dispatch of the same geometry allocates its
    // outputs for that many rows plus an eighth, launches its permute behind the layout and keeps the
    // result if the rows in use fit and fill at least four fifths of it; otherwise it permutes again
    // into exact outputs, as a first call of a geometry does.  Read and written with the mailbox held.
    struct OutputForecast {
        int64_t tokens = -1, topk = 0, experts = 0, alignment = 0, hidden = 0;
        bool expand = false;
        int64_t used_rows = 0;
    };
    int64_t forecast_rows(const OutputForecast& key) const {
        const OutputForecast& seen = forecast_;
        if (seen.tokens != key.tokens || seen.topk != key.topk || seen.experts != key.experts || seen.alignment != key.alignment ||
            seen.hidden != key.hidden || seen.expand != key.expand || seen.used_rows <= 0)
            return 0;
        return seen.used_rows + (seen.used_rows + 7) / 8;
    }
    void note_used_rows(OutputForecast key, int64_t used_rows) {
        key.used_rows = used_rows;
        forecast_ = key;
    }

    // Share of the routing choices that were valid in the latest fresh expanded dispatch, in 1/65536
    // (65536 before the first one).  A permute that is enqueued before the host knows the count sizes
    // its launch for this share of T * K plus half a percent instead of for all of it (a workgroup
    // that finds nothing to do costs about as much as one that takes a second turn, so the launch
    // aims at the count itself); any count is handled.
    int64_t valid_share_65536() const { return valid_share_65536_.load(); }
    void note_valid_share(int64_t assignments, int64_t choices) {
        if (choices > 0)
            valid_share_65536_.store((assignments * 65536 + choices - 1) / choices);
    }

    // The private handle tensors (slot table, slot-order list) of the latest few fresh expanded
    // dispatches.  A caller that keeps only the reference's seven handle tensors gets them back on
    // a replay of one of those handles: an entry is recognised by the identity of the handle's
    // routing snapshot (the tensor object, its data pointer and version) and of its recv_metadata
    // storage.  The two tensors are views of the allocation that backs the seven public ones.
    // Handles this runtime did not make, or made too long ago, are never matched: their replays
    // follow the handle's own recv_metadata and dst_slots in token order.
    void remember_private(const std::vector<torch::Tensor>& metadata, int64_t alignment) {
        if (metadata.size() < 9 || !metadata[7].defined() || !metadata[8].defined())
            return;
        RememberedHandle entry;
        entry.snapshot.emplace(metadata[5].getIntrusivePtr());
        entry.version = tensor_version(metadata[5]);
        entry.snapshot_data = metadata[5].data_ptr();
        entry.metadata_data = metadata[0].data_ptr();
        entry.rows = metadata[0].size(0);
        entry.alignment = alignment;
        entry.table = metadata[7];
        entry.order = metadata[8];
        std::vector<RememberedHandle> retired;  // released after the lock: a tensor's release may want the interpreter lock
        {
            std::lock_guard<std::mutex> lock(private_mutex_);
            // handles whose routing snapshot is gone can never come back
            for (auto it = remembered_.begin(); it != remembered_.end();) {
                if (it->snapshot->expired()) {
                    retired.push_back(std::move(*it));
                    it = remembered_.erase(it);
                } else {
                    ++it;
                }
            }
            remembered_.push_front(std::move(entry));
            while (remembered_.size() > kRememberedHandles) {
                retired.push_back(std::move(remembered_.back()));
                remembered_.pop_back();
            }
        }
    }

    // Appends the remembered private tensors to a seven-tensor handle when it is a remembered one
    // (alignment < 0: the caller does not know the handle's alignment, the identity decides).
    bool recall_private(std::vector<torch::Tensor>& metadata, int64_t alignment) const {
        std::lock_guard<std::mutex> lock(private_mutex_);
        if (closed_.load() || metadata.size() != 7)
            return false;
        for (const auto& entry : remembered_) {
            const auto alive = entry.snapshot->lock();
            if (!alive || alive.get() != metadata[5].unsafeGetTensorImpl() || metadata[5].data_ptr() != entry.snapshot_data ||
                tensor_version(metadata[5]) != entry.version || metadata[0].data_ptr() != entry.metadata_data ||
                metadata[0].size(0) != entry.rows || (alignment >= 0 && alignment != entry.alignment))
                continue;
            metadata.push_back(entry.table);
            metadata.push_back(entry.order);
            ++private_recalls_;
            return true;
        }
        return false;
    }

    // number of seven-tensor handles that got their private tensors back (for tests)
    int64_t private_recalls() const {
        std::lock_guard<std::mutex> lock(private_mutex_);
        return private_recalls_;
    }

    void forget_private() {
        std::deque<RememberedHandle> retired;
        std::array<std::shared_ptr<RebuiltHandle>, kRebuiltHandles> retired_rebuilt;
        std::lock_guard<std::mutex> lock(private_mutex_);
        retired.swap(remembered_);
        retired_rebuilt.swap(rebuilt_);
    }

    // The private tensors of a seven-tensor handle, rebuilt from the handle's own dst_slots and
    // recv_metadata (nanoep_rebuild_order) and kept for its later replays.  An entry is recognised
    // like a remembered one, and in addition by the identity and version of the two tensors it was
    // built from: a handle edited through torch is rebuilt.  `count` is where the device publishes the
    // number of list entries (tagged, so that a late store of an entry that used this word before is
    // never taken for this one's): until it is there, replays read the count on the device.
    struct RebuiltHandle {
        c10::weak_intrusive_ptr<c10::TensorImpl> snapshot;
        uint32_t snapshot_version = 0, metadata_version = 0, slots_version = 0;
        const void* snapshot_data = nullptr;
        const void* metadata_data = nullptr;
        const void* slots_data = nullptr;
        int64_t rows = 0, capacity = 0;
        torch::Tensor table, order;  // views of one allocation
        c10::Event ready{c10::DeviceType::CUDA};
        hipStream_t made_on = nullptr;
        int64_t* count = nullptr;  // pinned host word
        int64_t tag = 0;

        explicit RebuiltHandle(const torch::Tensor& snapshot_tensor) : snapshot(snapshot_tensor.getIntrusivePtr()) {}

        // the number of list entries once the device has published it, else -1
        int64_t published_entries() const {
            const int64_t word = __atomic_load_n(count, __ATOMIC_ACQUIRE);
            return word >= 0 && (word & ~int64_t{0xffffffff}) == tag ? (word & int64_t{0xffffffff}) : -1;
        }
    };

    std::shared_ptr<RebuiltHandle> find_rebuilt(const std::vector<torch::Tensor>& metadata, int64_t capacity) const {
        std::lock_guard<std::mutex> lock(private_mutex_);
        if (closed_.load() || metadata.size() != 7)
            return nullptr;
        for (const auto& entry : rebuilt_) {
            if (!entry)
                continue;
            const auto alive = entry->snapshot.lock();
            if (alive && alive.get() == metadata[5].unsafeGetTensorImpl() && metadata[5].data_ptr() == entry->snapshot_data &&
                tensor_version(metadata[5]) == entry->snapshot_version && metadata[0].data_ptr() == entry->metadata_data &&
                tensor_version(metadata[0]) == entry->metadata_version && metadata[3].data_ptr() == entry->slots_data &&
                tensor_version(metadata[3]) == entry->slots_version && metadata[0].size(0) == entry->rows && capacity == entry->capacity)
                return entry;
        }
        return nullptr;
    }

    // A new entry for this handle (tensors not yet set, not yet findable), with a count word and tag of
    // its own.  It takes the place of an entry whose handle is gone, else of the oldest one;
    // publish_rebuilt makes it findable once its tensors are there.
    std::shared_ptr<RebuiltHandle> new_rebuilt(const std::vector<torch::Tensor>& metadata, int64_t capacity) {
        auto entry = std::make_shared<RebuiltHandle>(metadata[5]);
        entry->snapshot_version = tensor_version(metadata[5]);
        entry->metadata_version = tensor_version(metadata[0]);
        entry->slots_version = tensor_version(metadata[3]);
        entry->snapshot_data = metadata[5].data_ptr();
        entry->metadata_data = metadata[0].data_ptr();
        entry->slots_data = metadata[3].data_ptr();
        entry->rows = metadata[0].size(0);
        entry->capacity = capacity;
        std::shared_ptr<RebuiltHandle> retired;  // released after the lock
        std::lock_guard<std::mutex> lock(private_mutex_);
        if (rebuilt_counts_ == nullptr) {  // (most runtimes never rebuild a handle, and pinned memory takes 40 us)
            void* words = nullptr;
            check_hip(hipHostMalloc(&words, kRebuiltHandles * sizeof(int64_t), hipHostMallocMapped | hipHostMallocCoherent), "hipHostMalloc");
            rebuilt_counts_ = static_cast<int64_t*>(words);
            for (size_t i = 0; i < kRebuiltHandles; ++i)
                rebuilt_counts_[i] = -1;
        }
        size_t at = kRebuiltHandles;
        for (size_t i = 0; i < kRebuiltHandles && at == kRebuiltHandles; ++i)
            if (!rebuilt_[i] || rebuilt_[i]->snapshot.expired())
                at = i;
        if (at == kRebuiltHandles)
            at = next_rebuilt_++ % kRebuiltHandles;
        entry->count = rebuilt_counts_ + at;
        entry->tag = (++rebuilt_generation_ & 0x3fffffff) << 32;
        retired = std::move(rebuilt_[at]);
        ++rebuilds_;
        return entry;
    }

    void publish_rebuilt(const std::shared_ptr<RebuiltHandle>& entry) {
        std::shared_ptr<RebuiltHandle> retired;  // released after the lock
        std::lock_guard<std::mutex> lock(private_mutex_);
        if (closed_.load())
            return;
        retired = std::move(rebuilt_[entry->count - rebuilt_counts_]);
        rebuilt_[entry->count - rebuilt_counts_] = entry;
    }

    // number of seven-tensor handles whose private tensors were rebuilt (for tests)
    int64_t rebuilds() const {
        std::lock_guard<std::mutex> lock(private_mutex_);
        return rebuilds_;
    }

    // Scratch of the layout kernels, kept between fresh dispatches (they take turns at the mailbox and
    // a turn ends when the layout has published its counts, but its last workgroups may still be reading
    // the scratch: the buffer is only handed out again to a call on the stream it was last used on,
    // where the launches are ordered; a call on another stream gets a buffer of its own, which is then
    // the one that is kept).  Called with the mailbox held.
    torch::Tensor layout_workspace(size_t bytes, hipStream_t stream, const c10::Device& device) {
        if (!workspace_.defined() || static_cast<size_t>(workspace_.numel()) < bytes || workspace_stream_ != stream) {
            workspace_ = new_tensor({static_cast<int64_t>(bytes)}, torch::kUInt8, device);
            workspace_stream_ = stream;
        }
        return workspace_;
    }

    // The stream for calls with a compute-unit budget below the whole device (the reference sizes its
    // cooperative grids with num_sms, csrc/pipeline.cu:20-24, so that communication kernels leave
    // compute units to the caller's own kernels; these kernels are sized by the work, so the budget
    // is enforced where the hardware offers it: a stream created with a CU mask).  Returns the raw
    // handle of a stream whose kernels run on about `cus` compute units, the same number on every
    // XCD; 0 when the budget is the whole device or the device's shape does not allow an even mask.
    // The streams are made on first use, shared by all runtimes of the process and never destroyed:
    // the caching allocator remembers the streams a block was used on and visits them when the block
    // is freed, which may be long after the buffer that used them is closed.
    //
    // Which mask bit is which CU differs between descriptions of the interface (bit i on XCD i mod N,
    // or XCDs one after the other), so the mask is one that gives every XCD the same number of CUs
    // under both readings: with N XCDs of P CUs, bit P*a + N*b + c is set when (a + c) mod N < t.
    // That confines the budget to steps of P (32 of 256 on an MI355X), rounded down, at least one step.
    int64_t budget_stream(int cus) {
        TORCH_CHECK(!closed_.load(), "PeerRuntime is closed");
        DeviceGuard guard(static_cast<c10::DeviceIndex>(device_));  // (the topology is the current device's)
        int device_cus = 0, xcds = 0;
        check_status(nanoep_device_topology(&device_cus, &xcds, nullptr), "device_topology");
        if (cus <= 0 || cus >= device_cus || xcds <= 1 || device_cus % xcds != 0 || (device_cus / xcds) % xcds != 0)
            return 0;
        const int per_xcd = device_cus / xcds;
        const int steps = std::max(1, cus / per_xcd);  // of `per_xcd` CUs each: per_xcd / xcds on every XCD
        if (steps >= xcds)
            return 0;
        static std::mutex streams_mutex;
        static std::vector<std::tuple<int, int, hipStream_t>> streams;  // (device, steps, stream)
        std::lock_guard<std::mutex> lock(streams_mutex);
        for (const auto& made : streams)
            if (std::get<0>(made) == device_ && std::get<1>(made) == steps)
                return reinterpret_cast<int64_t>(std::get<2>(made));
        std::vector<uint32_t> mask((device_cus + 31) / 32, 0u);
        for (int bit = 0; bit < device_cus; ++bit) {
            const int a = bit / per_xcd, c = bit % xcds;
            if ((a + c) % xcds < steps)
                mask[bit / 32] |= 1u << (bit % 32);
        }
        hipStream_t stream = nullptr;
        check_hip(hipExtStreamCreateWithCUMask(&stream, static_cast<uint32_t>(mask.size()), mask.data()), "hipExtStreamCreateWithCUMask");
        streams.emplace_back(device_, steps, stream);
        return reinterpret_cast<int64_t>(stream);
    }

    // compute units a budget stream's kernels can run on (what budget_stream rounds `cus` to)
    int budget_stream_cus(int cus) const {
        DeviceGuard guard(static_cast<c10::DeviceIndex>(device_));
        int device_cus = 0, xcds = 0;
        check_status(nanoep_device_topology(&device_cus, &xcds, nullptr), "device_topology");
        if (cus <= 0 || cus >= device_cus || xcds <= 1 || device_cus % xcds != 0 || (device_cus / xcds) % xcds != 0)
            return device_cus;
        const int per_xcd = device_cus / xcds;
        const int steps = std::max(1, cus / per_xcd);
        return steps >= xcds ? device_cus : steps * per_xcd;
    }

    py::bytes export_local_handle() const {
        std::string tag(64, '\0');
        tag.replace(0, 9, "nanoep-r1");
        return py::bytes(tag);
    }

    void import_peer_handles(const std::vector<py::bytes>& handles) {
        TORCH_CHECK(!closed_.load(), "PeerRuntime is closed");
        if (handles.size() != 1)
            throw py::value_error("expected exactly one handle (world_size == 1)");
        for (const auto& handle : handles)
            if (py::len(handle) != 64)
                throw py::value_error("Each IPC handle must contain exactly 64 bytes");
        mappings_closed_ = false;
    }

    torch::Tensor local_window() {
        TORCH_CHECK(!closed_.load(), "PeerRuntime is closed");
        if (!window_.defined()) {
            DeviceGuard guard(static_cast<c10::DeviceIndex>(device_));
            window_ = torch::zeros({num_bytes_}, torch::dtype(torch::kUInt8).device(torch::kCUDA, device_));
        }
        return window_;
    }

    torch::Tensor peer_addresses() {
        auto window = local_window();
        auto addresses = torch::empty({1}, torch::dtype(torch::kInt64));
        addresses[0] = reinterpret_cast<int64_t>(window.data_ptr());
        return addresses.to(window.device());
    }

    // No peers: an epoch barrier has nobody to meet.  Epochs still have to increase, as in the
    // reference (csrc/peer.cu:234-237).
    void barrier(int64_t) {
        require_usable();
        ++last_barrier_epoch_;
    }
    void barrier_at(int64_t, int64_t epoch) {
        require_usable();
        TORCH_CHECK(epoch > last_barrier_epoch_, "Barrier epoch must strictly increase");
        last_barrier_epoch_ = epoch;
    }

    void close_peer_mappings() {
        if (closed_.load() || mappings_closed_)
            return;
        TORCH_CHECK(!counts_pending_.load(), "Cannot close while a fresh dispatch is waiting for counts");
        mappings_closed_ = true;
    }

    void close() {
        if (closed_.load())
            return;
        TORCH_CHECK(mappings_closed_, "Call close_peer_mappings() before close()");
        window_ = torch::Tensor();
        forget_private();

        {
            std::lock_guard<std::mutex> lock(counts_mutex_);
            workspace_ = torch::Tensor();
        }
        closed_.store(true);
    }

   private:
    struct RememberedHandle {
        std::optional<c10::weak_intrusive_ptr<c10::TensorImpl>> snapshot;
        uint32_t version = 0;
        const void* snapshot_data = nullptr;
        const void* metadata_data = nullptr;
        int64_t rows = 0;
        int64_t alignment = 0;
        torch::Tensor table, order;
    };

    // in-place edits through torch bump the version; inference tensors have none
    static uint32_t tensor_version(const torch::Tensor& tensor) {
        return tensor.is_inference() ? 0u : tensor.unsafeGetTensorImpl()->version_counter().current_version();
    }

    int device_ = 0;
    int64_t num_bytes_ = 0;
    int64_t* host_counts_ = nullptr;
    torch::Tensor window_;
    std::mutex counts_mutex_;
    std::atomic<bool> counts_pending_{false};
    std::atomic<bool> counts_failed_{false};
    std::atomic<bool> prefers_exact_outputs_{false};
    OutputForecast forecast_;
    std::atomic<int64_t> valid_share_65536_{65536};
    std::deque<RememberedHandle> remembered_;  // newest first
    std::array<std::shared_ptr<RebuiltHandle>, kRebuiltHandles> rebuilt_;
    int64_t* rebuilt_counts_ = nullptr;  // pinned, one word per entry of rebuilt_
    size_t next_rebuilt_ = 0;
    int64_t rebuilt_generation_ = 0;
    int64_t rebuilds_ = 0;
    torch::Tensor workspace_;
    hipStream_t workspace_stream_ = nullptr;
    mutable int64_t private_recalls_ = 0;
    mutable std::mutex private_mutex_;
    int64_t last_barrier_epoch_ = 0;
    bool mappings_closed_ = false;
    std::atomic<bool> closed_{false};
};

// What a caller gets back from an asynchronous call: a marker on the communication stream behind
// the call's kernels, and the tensors those kernels read and write (the role of
// csrc/include/nano_ep/event.hpp:12-28 in the reference).  Waiting puts the consumer's stream behind the
// marker.
//
// The marker holds the tensors until somebody has waited, so that none of them is freed while the
// kernels use it on a stream its allocator does not know of; waiting tells the allocator of the
// consumer's stream instead, which costs nothing for tensors that were allocated there (telling it of the
// communication stream makes it record an event for every block when it is freed).  A marker that goes
// away with nobody having waited tells it of the communication stream after all.  It is made before
// the call enqueues anything, so that this also covers a call that ends in an error half way: bad routing
// ids are known while the layout and the permute behind it are still at work.  A synchronous call with a
// compute-unit budget has a marker for that alone.
//
// A caller that is on the communication stream itself most likely waits there, and gets an event: on one
// queue that is no work for the GPU, where the store of a StreamPoint stands between the kernels (8192 x 2048
// top-8, alignment 128, launch period: event 55.2 us a dispatch and 50.5 a combine, store 59.4 and 55.2).
class CompletionEvent {
   public:
    explicit CompletionEvent(const Stream& producer) : done_(c10::DeviceType::CUDA), producer_(producer) {}
    CompletionEvent(const CompletionEvent&) = delete;
    CompletionEvent& operator=(const CompletionEvent&) = delete;
    ~CompletionEvent() {
        if (settled_)
            return;
        try {
            note_use(written_, producer_);
            note_use(read_, producer_);
        } catch (...) {
        }
    }

    // What the call's kernels read, and what they write: held from before they are enqueued.
    void reads(const torch::Tensor& tensor) { read_.push_back(tensor); }
    void reads(const std::vector<torch::Tensor>& tensors) { read_.insert(read_.end(), tensors.begin(), tensors.end()); }
    void writes(const torch::Tensor& tensor) { written_.push_back(tensor); }

    // What was written so far is no result after all: in use for as long as what is read.
    void discard_written() {
        reads(written_);
        written_.clear();
    }

    // The call is complete: the marker goes behind all that its stream holds now.
    void record(const Stream& caller) {
        if (producer_.stream() != caller.stream() && !capturing(producer_))
            point_ = StreamPoints::of(producer_.device_index()).record(producer_);
        if (!point_.has_value())
            done_.record(producer_.unwrap());
    }

    // The caller's stream has come behind the work without this marker: the tensors need nobody any more.
    void settle() { settled_ = true; }

    void order_after(const Stream& consumer) {
        std::vector<torch::Tensor> let_go;  // behind the lock: a tensor's end may run Python, and that other waiters of this marker
        std::lock_guard<std::mutex> lock(mutex_);
        if (point_.has_value() && !capturing(consumer)) {
            if (!point_->reached())
                StreamPoints::wait(consumer, *point_);
        } else {
            // A consumer under capture is told of an event, and the runtime says what it makes of that.
            if (point_.has_value())
                done_.record(producer_.unwrap());
            consumer.unwrap().wait(done_);
        }
        note_use(written_, consumer);
        note_use(read_, consumer);
        let_go.swap(read_);
        settled_ = true;
    }

    void current_stream_wait() { order_after(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA()); }

   private:
    static void note_use(const std::vector<torch::Tensor>& tensors, const Stream& stream) {
        for (const auto& tensor : tensors)
            if (tensor.defined() && tensor.numel() > 0)
                tensor.record_stream(stream.unwrap());
    }

    std::mutex mutex_;
    std::optional<StreamPoint> point_;
    c10::Event done_;  // where there is no point, or a consumer under capture
    Stream producer_;
    bool settled_ = false;  // somebody has waited, or nobody needs to
    std::vector<torch::Tensor> written_, read_;
};

namespace {

// What a tensor argument has to look like: where it lives, its element type and its extents
// (-1 leaves an extent open).  Every tensor check of dispatch, combine and the cached handle is one
// `require`; the message is the caller-visible part.
bool describes(const torch::Tensor& tensor, const c10::Device& device, at::ScalarType dtype, std::initializer_list<int64_t> extents) {
    if (!tensor.defined() || tensor.device() != device || tensor.scalar_type() != dtype || !tensor.is_contiguous() ||
        tensor.dim() != static_cast<int64_t>(extents.size()))
        return false;
    const auto sizes = tensor.sizes();
    size_t axis = 0;
    for (const int64_t extent : extents) {
        if (extent >= 0 && sizes[axis] != extent)
            return false;
        ++axis;
    }
    return true;
}

template <class... Message>
void require(const torch::Tensor& tensor, const c10::Device& device, at::ScalarType dtype, std::initializer_list<int64_t> extents,
             const Message&... message) {
    TORCH_CHECK(describes(tensor, device, dtype, extents), message...);
}

bool vector_aligned(const torch::Tensor& tensor) {
    return tensor.numel() == 0 || reinterpret_cast<uintptr_t>(tensor.data_ptr()) % 16 == 0;
}

// The payload, its routing ids and its weights, as the reference's host pipeline insists on them
// (csrc/pipeline.cu:26-60): same limits, same wording of what is wrong.
void require_dispatch_inputs(const torch::Tensor& x, const torch::Tensor& routing, const c10::optional<torch::Tensor>& weights,
                             int device, int64_t num_experts, int64_t max_tokens) {
    const c10::Device here(c10::DeviceType::CUDA, static_cast<c10::DeviceIndex>(device));
    TORCH_CHECK(x.defined() && x.is_cuda() && x.device() == here && x.dim() == 2 && x.is_contiguous(),
                "x must be contiguous CUDA [T,H] on the runtime device");
    require(x, here, torch::kBFloat16, {-1, -1}, "dispatch x must be bfloat16");
    const int64_t tokens = x.size(0), hidden = x.size(1);
    TORCH_CHECK(hidden > 0 && hidden % kHiddenAlignment == 0, "dispatch hidden must be a positive multiple of 256");
    TORCH_CHECK(vector_aligned(x), "dispatch x data pointer must be 16-byte aligned");
    require(routing, here, torch::kInt64, {tokens, -1}, "indices must be contiguous CUDA int64 [T,K] on the x device");
    const int64_t topk = routing.size(1);
    TORCH_CHECK(topk >= 1 && topk <= 32, "num_topk must be in [1, 32]");
    TORCH_CHECK(num_experts > 0, "num_experts must be positive and divisible by world_size");
    TORCH_CHECK(max_tokens <= std::numeric_limits<int32_t>::max(), "max_tokens exceeds int32 metadata range");
    TORCH_CHECK(max_tokens > 0 && tokens <= max_tokens, "source token count exceeds max_tokens");
    if (weights.has_value())
        require(*weights, here, torch::kFloat32, {tokens, topk}, "weights must be contiguous CUDA float32 [T,K] on the x device");
}

// The seven handle tensors of a cached call against the geometry they must describe.
void require_handle_tensors(const std::vector<torch::Tensor>& metadata, const c10::Device& here, int64_t source_tokens, int64_t topk,
                            int64_t local_experts) {
    const auto field = [&](int index, const char* name, at::ScalarType dtype, std::initializer_list<int64_t> extents) {
        require(metadata[index], here, dtype, extents, "cached ", name, " has invalid CUDA storage or shape");
    };
    field(0, "recv_metadata", torch::kInt32, {-1, topk + 2});
    field(1, "expert_counts", torch::kInt64, {local_experts});
    field(2, "expert_offsets", torch::kInt64, {local_experts + 1});
    field(3, "dst_slots", torch::kInt64, {source_tokens, 1});
    field(4, "send_counts", torch::kInt64, {1});
    field(5, "source_topk_snapshot", torch::kInt64, {source_tokens, topk});
    field(6, "recv_rank_prefix", torch::kInt64, {1});
}

// The optional eighth handle tensor: int32 [T,K] slot table written by the layout kernels.
const int32_t* slot_table(const std::vector<torch::Tensor>& metadata, int64_t tokens, int64_t topk, bool expand) {
    if (!expand || metadata.size() < 8 || !metadata[7].defined())
        return nullptr;
    const auto& table = metadata[7];
    TORCH_CHECK(table.device() == metadata[0].device() && table.scalar_type() == torch::kInt32 && table.is_contiguous() &&
                    table.dim() == 2 && table.size(0) == tokens && table.size(1) == topk,
                "cached slot table has invalid CUDA storage or shape");
    return table.numel() == 0 ? nullptr : table.data_ptr<int32_t>();
}

// The optional ninth handle tensor: int64 slot-order list written by the layout kernels.
const int64_t* slot_order_list(const std::vector<torch::Tensor>& metadata, int64_t tokens, int64_t topk, int64_t local_experts,
                               bool expand, int64_t* entries) {
    *entries = 0;
    if (!expand || metadata.size() < 9 || !metadata[8].defined())
        return nullptr;
    const auto& order = metadata[8];
    TORCH_CHECK(order.device() == metadata[0].device() && order.scalar_type() == torch::kInt64 && order.is_contiguous() &&
                    order.dim() == 1 && order.size(0) <= nanoep_slot_order_entries(tokens, static_cast<int>(topk), local_experts),
                "cached slot-order list has invalid CUDA storage or shape");
    // the whole buffer (list + count word) defers to the count on the device
    const bool whole = order.numel() > 0 && order.numel() == nanoep_slot_order_entries(tokens, static_cast<int>(topk), local_experts);
    *entries = whole ? -1 : order.numel();
    return order.numel() == 0 ? nullptr : order.data_ptr<int64_t>();
}

// Communication stream waits for the producer of the inputs: the caller's stream, an explicit
// event, or both (csrc/pipeline.cu:364-377 in the reference).
// An external-stream wrapper never compares equal to a pool stream object, so identity is decided
// on the raw handles: when the caller already runs on the communication stream no event is needed.
bool same_queue(const Stream& a, const Stream& b) { return a.stream() == b.stream(); }

// Stream the kernels are enqueued on.  An asynchronous call uses the buffer's communication stream.
// A synchronous call must leave its results ordered on the caller's stream, so it runs there
// directly instead of bouncing through the communication stream with two cross-stream events; it
// still comes after everything enqueued earlier on the communication stream.
//
// kNoStream in place of that stream says that nothing has ever been put on it: a synchronous call then has
// nothing there to come behind, and a stream that nobody uses is never set up (the handle alone takes
// the runtime 80 us, the first question how it is doing 120 to 200 us, of a new buffer's first call).
constexpr int64_t kNoStream = -1;

Stream work_stream(int64_t comm_handle, const Stream& compute, c10::DeviceIndex device, bool async_op, bool budgeted) {
    if (comm_handle == kNoStream) {
        TORCH_CHECK(!async_op && !budgeted, "an asynchronous call, or one with a compute-unit budget, needs its stream");
        return compute;
    }
    const auto comm = external_stream(comm_handle, device);
    // (a call with a compute-unit budget runs on the stream it was handed: that stream carries the CU mask)
    if (async_op || budgeted || same_queue(comm, compute))
        return comm;
    // While the caller's stream is being captured into a graph no other stream may be queried;
    // a captured call is ordered by the graph alone.  A communication stream under capture holds nothing that runs
    // before its graph does: waiting for it would make the call part of that graph.
    if (!capturing(compute) && !capturing(comm) && busy(comm))
        wait_on(compute, comm);
    return compute;
}

// Makes `stream` the current one of its device while it lives, if it is another one than `current`.
class StreamSwitch {
   public:
    StreamSwitch(const Stream& stream, const Stream& current) {
        if (!same_queue(stream, current))
            guard_.reset_stream(stream.unwrap());
    }

   private:
    OptionalStreamGuard guard_;
};

void order_comm_after_inputs(const Stream& comm, const Stream& compute, int64_t previous_event, bool async_op) {
    if (previous_event != -1) {
        if (!async_op && !same_queue(comm, compute))
            wait_on(comm, compute);
        check_hip(hipStreamWaitEvent(comm.stream(), reinterpret_cast<hipEvent_t>(previous_event), 0), "hipStreamWaitEvent");
    } else if (!same_queue(comm, compute)) {
        wait_on(comm, compute);
    }
}

// The private tensors of a seven-tensor expanded handle the runtime does not remember: found among
// the ones rebuilt earlier, or rebuilt now on `stream` (the current stream of the allocator).
std::shared_ptr<PeerRuntime::RebuiltHandle> private_tensors_of(PeerRuntime& runtime, const std::vector<torch::Tensor>& metadata,
                                                               int64_t capacity, int64_t tokens, int64_t topk, int64_t local_experts,
                                                               int64_t hidden, const Stream& stream) {
    auto entry = runtime.find_rebuilt(metadata, capacity);
    if (entry) {
        if (entry->made_on != stream.stream()) {
            // built on another stream: wait for it unless it is long done, and tell the allocator
            if (!entry->ready.query())
                stream.unwrap().wait(entry->ready);
            entry->order.record_stream(stream.unwrap());  // the table is a view of the same allocation
        }
        return entry;
    }
    entry = runtime.new_rebuilt(metadata, capacity);
    const int64_t order_words = nanoep_slot_order_entries(tokens, static_cast<int>(topk), local_experts);
    const size_t workspace_bytes = nanoep_rebuild_workspace_bytes(tokens, static_cast<int>(topk));
    const int64_t table_words = (tokens * topk + 1) / 2;
    const int64_t workspace_words = static_cast<int64_t>((workspace_bytes + 7) / 8);
    // one allocation: slot-order buffer | slot table | the rebuild's scratch
    auto storage = torch::empty({order_words + table_words + workspace_words}, metadata[3].options());
    entry->order = storage.narrow(0, 0, order_words);
    entry->table = storage.narrow(0, order_words, table_words).view(torch::kInt32).narrow(0, 0, tokens * topk).view({tokens, topk});
    check_status(nanoep_rebuild_order(metadata[0].data_ptr<int32_t>(), metadata[3].data_ptr<int64_t>(), metadata[0].size(0), capacity, tokens,
                                      static_cast<int>(topk), local_experts, static_cast<int>(hidden), entry->table.data_ptr<int32_t>(),
                                      entry->order.data_ptr<int64_t>(), storage.data_ptr<int64_t>() + order_words + table_words,
                                      static_cast<size_t>(workspace_words) * 8, entry->count, entry->tag, stream.stream()),
                 "rebuild_order");
    entry->made_on = stream.stream();
    entry->ready.record(stream.unwrap());
    runtime.publish_rebuilt(entry);
    return entry;
}

}  // namespace

using DispatchResult =
    std::tuple<std::vector<torch::Tensor>, std::vector<torch::Tensor>, std::array<int64_t, 2>, std::shared_ptr<CompletionEvent>>;

DispatchResult dispatch(PeerRuntime& runtime,
                        const torch::Tensor& x,
                        const torch::Tensor& indices,
                        const c10::optional<torch::Tensor>& weights,
                        int64_t num_experts,
                        int64_t max_tokens,
                        int64_t alignment,
                        const std::vector<torch::Tensor>& cached_metadata,
                        int64_t cached_expanded_capacity,
                        bool /*allow_multiple_reduction*/,
                        bool expand,
                        bool zero_padding,
                        int num_sms,
                        int64_t comm_stream,
                        int64_t previous_event,
                        bool async_op) {
    const bool cached = !cached_metadata.empty();
    TORCH_CHECK(!cached || (cached_metadata.size() >= 7 && cached_metadata.size() <= 9),
                "cached metadata must contain the seven prepared tensors from dispatch (plus the optional slot table and slot-order list)");
    const auto& routing = cached ? cached_metadata[5] : indices;
    runtime.require_usable();
    require_dispatch_inputs(x, routing, weights, runtime.device(), num_experts, max_tokens);
    TORCH_CHECK(alignment > 0, "alignment must be positive");
    const auto device = static_cast<c10::DeviceIndex>(runtime.device());
    DeviceGuard device_guard(device);
    const int cu_budget = resolve_cu_budget(num_sms, device);

    const int64_t tokens = x.size(0);
    const int64_t hidden = x.size(1);
    const int64_t topk = routing.size(1);
    const int64_t local_experts = num_experts;

    const auto compute = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device);
    const auto comm = work_stream(comm_stream, compute, device, async_op, cu_budget != 0);
    const StreamSwitch on_comm(comm, compute);
    // Answers for what the call uses on a stream that the memory's owner may not know of.
    const auto marker = async_op || !same_queue(comm, compute) ? std::make_shared<CompletionEvent>(comm) : nullptr;
    if (marker) {
        marker->reads(x);
        if (cached)
            marker->reads(cached_metadata);
        else
            marker->reads(indices);
        if (weights.has_value())
            marker->reads(*weights);
    }
    // Results are allocated on the caller's stream: the work is ordered behind what that stream holds
    // then, and what it does with the results comes behind the call (a synchronous one) or
    // behind the completion event, which holds them until somebody has waited.  An asynchronous call with
    // an event of its own is ordered behind that event only: its results come from the communication
    // stream's pool.
    //
    // The caller's stream may be other threads' as well: a block of its pool may have been freed a moment ago, with the
    // kernels that used it still to run.  So the communication stream comes behind the caller's
    // after the allocation, never before it; one that has to be made later is followed by a wait of its own.
    const bool callers_pool = !async_op || previous_event == -1;
    const bool borrows = callers_pool && !same_queue(comm, compute);
    const c10::Device here = x.device();
    torch::Tensor out_x, out_indices, out_weights;
    // x_rows rows of payload (and expanded weights), n_rows rows of compact indices / weights
    const auto allocate_outputs = [&](int64_t x_rows, int64_t n_rows) {
        const StreamSwitch pool(callers_pool ? compute : comm, comm);
        out_x = new_tensor({x_rows, hidden}, torch::kBFloat16, here);
        if (!expand)
            out_indices = new_tensor({n_rows, topk}, torch::kInt64, here);
        if (weights.has_value())
            out_weights = expand ? new_tensor({x_rows}, torch::kFloat32, here) : new_tensor({n_rows, topk}, torch::kFloat32, here);
        if (marker)
            for (const auto* tensor : {&out_x, &out_indices, &out_weights})
                marker->writes(*tensor);
    };
    // What the permute reads of a handle, as plain pointers.  order_entries: A, or -1 for "the whole
    // slot-order buffer is there and the kernel finds A in its last word".
    struct HandleView {
        const int32_t* recv_metadata = nullptr;
        const int64_t* dst_slots = nullptr;
        const int32_t* token_slots = nullptr;
        const int64_t* slot_order = nullptr;
        int64_t order_entries = 0;
        const int64_t* expert_counts = nullptr;
        const int64_t* expert_offsets = nullptr;
    };
    const auto view_of = [&](const std::vector<torch::Tensor>& handle) {
        HandleView view;
        view.recv_metadata = handle[0].data_ptr<int32_t>();
        view.dst_slots = handle[3].data_ptr<int64_t>();
        view.token_slots = slot_table(handle, tokens, topk, expand);
        view.slot_order = slot_order_list(handle, tokens, topk, local_experts, expand, &view.order_entries);
        view.expert_counts = handle[1].data_ptr<int64_t>();
        view.expert_offsets = handle[2].data_ptr<int64_t>();
        return view;
    };
    // count_on_device: the number of list entries in use is not known on the host yet
    const auto launch_permute = [&](HandleView handle, int64_t received, int64_t capacity, bool count_on_device = false) {
        TORCH_CHECK(!count_on_device || handle.slot_order == nullptr || handle.order_entries == -1, "slot-order buffer is incomplete");
        if (count_on_device && handle.slot_order != nullptr) {
            // the launch is sized for the share of valid choices the runtime saw last, plus 0.5 %
            const int64_t share = runtime.valid_share_65536() + 328;
            const int64_t expected = share >= 65536 ? tokens * topk : tokens * topk * share / 65536;
            handle.order_entries = expected >= tokens * topk || expected < 2 ? -1 : -expected;
        }
        check_status(
            nanoep_dispatch(x.data_ptr(), weights.has_value() ? weights->data_ptr<float>() : nullptr, handle.recv_metadata, handle.dst_slots,
                            handle.token_slots, handle.slot_order, handle.order_entries, handle.expert_counts, handle.expert_offsets,
                            received, capacity, tokens, static_cast<int>(hidden), static_cast<int>(topk), local_experts, alignment,
                            expand ? 1 : 0, zero_padding ? 1 : 0, out_x.data_ptr(), expand ? nullptr : out_indices.data_ptr<int64_t>(),
                            weights.has_value() ? out_weights.data_ptr<float>() : nullptr, cu_budget, comm.stream()),
            "dispatch");
    };

    std::vector<torch::Tensor> metadata;
    int64_t recv_count = 0;
    int64_t expanded_capacity = 0;
    if (cached) {
        require_handle_tensors(cached_metadata, x.device(), tokens, topk, local_experts);
        metadata = cached_metadata;
        recv_count = cached_metadata[0].size(0);
        expanded_capacity = cached_expanded_capacity;
        TORCH_CHECK(recv_count <= tokens && expanded_capacity >= 0, "cached handle does not match the payload");
        TORCH_CHECK(!expand || expanded_capacity <= std::numeric_limits<int32_t>::max(),
                    "expanded capacity exceeds int32 metadata range");
        allocate_outputs(expand ? expanded_capacity : recv_count, recv_count);
        order_comm_after_inputs(comm, compute, previous_event, async_op);
        // A handle that went through the reference's Python class carries the seven tensors of the
        // reference only.  If it is one of this runtime's latest fresh dispatches, the runtime still
        // has its private tensors and the payload takes the slot-order walk
        // (the RECALL_ORDER switch set to 0 turns that off).  Any other seven-tensor handle is followed as it
        // is written, in token order through its own dst_slots and recv_metadata: whatever row and
        // slot order it describes is the order the rows land in.
        bool has_private = metadata.size() > 7;
        if (expand && recv_count > 0 && !has_private && tuning_switch("RECALL_ORDER") != 0)
            has_private = runtime.recall_private(metadata, alignment);
        if (recv_count > 0) {
            HandleView view = view_of(metadata);
            // A seven-tensor handle the runtime does not remember: its private tensors are rebuilt from
            // the handle as it is written (one integer pass, two launches) and kept for its later
            // replays, where the payload is large enough for the slot-order walk to pay for that
            // (the REBUILD_ORDER switch: 0 never, 1 always).  Not under stream capture: a captured
            // replay must not depend on when the rebuilt tensors are dropped.
            const int rebuild_switch = expand && !has_private ? tuning_switch("REBUILD_ORDER") : 0;
            const bool worth_it = rebuild_switch >= 0 ? rebuild_switch != 0 : expanded_capacity * hidden * 2 >= kRebuildPayloadBytes;
            std::shared_ptr<PeerRuntime::RebuiltHandle> rebuilt;
            if (expand && !has_private && worth_it && tokens * topk < (int64_t{1} << 31) &&
                nanoep_slot_order_entries(tokens, static_cast<int>(topk), local_experts) > 0) {
                if (!capturing(comm))
                    rebuilt = private_tensors_of(runtime, metadata, expanded_capacity, tokens, topk, local_experts, hidden, comm);
            }
            if (rebuilt) {
                view.token_slots = rebuilt->table.data_ptr<int32_t>();
                view.slot_order = rebuilt->order.data_ptr<int64_t>();
                const int64_t entries = rebuilt->published_entries();
                view.order_entries = entries >= 0 ? entries : -1;
            }
            launch_permute(view, recv_count, expanded_capacity, /*count_on_device=*/rebuilt && view.order_entries < 0);
        }
    } else {
        // the slot-order list packs token * K + k into 32 bits
        const bool ordered = expand && tokens * topk < (int64_t{1} << 31);
        // The handle tensors of one call are views of one allocation (the int64 ones, then the int32 ones), and the
        // views are made after the layout has been enqueued: on a path whose small-batch cost is
        // host latency, the GPU starts three allocator round trips after the call instead of ten
        // and works while the rest of the bookkeeping is done.
        const int64_t order_entries = ordered ? nanoep_slot_order_entries(tokens, static_cast<int>(topk), local_experts) : 0;
        // offsets of the int64 tensors in the arena; the per-token ones start 16-byte aligned (even offsets)
        const auto even = [](int64_t words) { return (words + 1) / 2 * 2; };
        const int64_t at_offsets = local_experts, at_send = 2 * local_experts + 1, at_prefix = at_send + 1;
        const int64_t at_dst = even(at_prefix + 1), at_snapshot = even(at_dst + tokens), at_order = even(at_snapshot + tokens * topk);
        const int64_t count64 = even(at_order + order_entries);
        const int64_t at_table = (tokens * (topk + 2) + 3) / 4 * 4;  // the slot table starts 16-byte aligned
        const int64_t count32 = at_table + (expand ? tokens * topk : 0);
        const size_t workspace_bytes = nanoep_layout_workspace_bytes(tokens, static_cast<int>(topk), local_experts);
        TORCH_CHECK(workspace_bytes > 0, "unsupported routing geometry for the layout kernels");
        TORCH_CHECK(nanoep_layout_block_tokens(tokens, local_experts, static_cast<int>(hidden)) > 0,
                    "the layout kernels take at most 3839 local experts, got ", local_experts);
        // one allocation: the int64 tensors first, the int32 ones behind them as a view of the same storage
        torch::Tensor arena;
        {
            const StreamSwitch pool(callers_pool ? compute : comm, comm);
            arena = new_tensor({count64 + (count32 + 1) / 2}, torch::kInt64, here);
        }
        if (marker)
            marker->writes(arena);
        // int64: expert_counts [L] | expert_offsets [L+1] | send_counts [1] | recv_rank_prefix [1] |
        //        dst_slots [T] | topk snapshot [T*K] | slot_order;   int32: recv_metadata [T*(K+2)] | token_slots [T*K]
        int64_t* base64 = arena.data_ptr<int64_t>();
        int32_t* base32 = reinterpret_cast<int32_t*>(base64 + count64);

        // From here until the counts have been read this call owns the runtime's mailbox; a fresh
        // dispatch of another thread on the same runtime waits here for its turn.
        PeerRuntime::CountsTurn turn(runtime);

        // The exact shapes (N, C) are only known once the layout kernels have run.  Waiting for
        // them before launching the permute leaves the GPU idle for a host round trip, so where the
        // upper bound of the shapes (every choice valid plus every expert's worst alignment gap) is
        // close to what routing will fill, the outputs are allocated at that bound, the permute is
        // enqueued right behind the layout and the results are narrowed afterwards.  "Close" is
        // kept honest in both directions: the gaps may add at most an eighth to the bound, and a call
        // that still ends up holding more than 1.25 times the rows it uses (many masked choices)
        // permutes again into exact outputs and turns the runtime to the exact order, in which the
        // outputs are allocated after the counts are known, until a call shows the bound close again.
        const int64_t choice_bound = expand ? tokens * topk : tokens;
        const int64_t gap_bound = expand ? local_experts * (alignment - 1) : 0;
        const int64_t row_bound = choice_bound + gap_bound;
        const bool bound_rule = gap_bound * 8 <= choice_bound;
        PeerRuntime::OutputForecast geometry;
        geometry.tokens = tokens, geometry.topk = topk, geometry.experts = local_experts, geometry.alignment = alignment;
        geometry.hidden = hidden, geometry.expand = expand;
        // rows the outputs are allocated for ahead of the counts: the bound where it is close, else what
        // the latest call of this geometry used plus an eighth, else nothing (the exact order)
        const auto rows_ahead = [&]() -> int64_t {
            const int order_switch = tuning_switch("FRESH_OUTPUTS");  // 0: always exact, 1: at the bound whenever the rule allows it
            if (tokens == 0 || order_switch == 0 || row_bound > std::numeric_limits<int32_t>::max())
                return 0;
            if (!bound_rule)
                return std::min(row_bound, runtime.forecast_rows(geometry));
            return order_switch == 1 || !runtime.prefers_exact_outputs() ? row_bound : 0;
        };
        int64_t early_rows = 0;
        if (borrows && (early_rows = rows_ahead()) > 0)
            allocate_outputs(early_rows, tokens);
        order_comm_after_inputs(comm, compute, previous_event, async_op);
        TORCH_CHECK(!capturing(comm), "Fresh dispatch with host count polling cannot be captured in a HIP graph");

        const auto workspace = runtime.layout_workspace(workspace_bytes, comm.stream(), here);
        turn.begin();
        const int layout_status =
            nanoep_layout_ahead(routing.data_ptr<int64_t>(), tokens, static_cast<int>(topk), local_experts, alignment, expand ? 1 : 0,
                                static_cast<int>(hidden), base32, base64, base64 + at_offsets, base64 + at_dst, base64 + at_send,
                                base64 + at_snapshot, base64 + at_prefix, expand ? base32 + at_table : nullptr,
                                order_entries > 0 ? base64 + at_order : nullptr, workspace.data_ptr(), workspace_bytes, turn.mailbox(),
                                tokens > 0 ? x.data_ptr() : nullptr, comm.stream());
        if (layout_status != NANOEP_OK && layout_status != NANOEP_ERR_HIP)
            turn.abandon();  // refused before anything was enqueued
        check_status(layout_status, "layout");

        if (!borrows)  // (off the path to the layout)
            early_rows = rows_ahead();
        const bool speculative = early_rows > 0;
        if (speculative) {
            // enqueued straight from the arena's pointers: the tensors of the handle are made below,
            // while the GPU works
            HandleView fresh;
            fresh.recv_metadata = base32;
            fresh.dst_slots = base64 + at_dst;
            fresh.token_slots = expand ? base32 + at_table : nullptr;
            fresh.slot_order = order_entries > 0 ? base64 + at_order : nullptr;
            fresh.order_entries = order_entries > 0 ? -1 : 0;
            fresh.expert_counts = base64;
            fresh.expert_offsets = base64 + at_offsets;
            try {
                if (!borrows)
                    allocate_outputs(early_rows, tokens);
                launch_permute(fresh, tokens, early_rows, /*count_on_device=*/true);
            } catch (...) {
                // The layout is under way and will publish its counts whatever went wrong here (most
                // likely the allocation at the bound): the turn at the mailbox is settled before the
                // error leaves, so the runtime stays usable.  Only counts that never arrive latch it.
                int64_t unused[NANOEP_HOST_COUNT_WORDS] = {0, 0, 0, 0};
                try {
                    turn.wait(comm.stream(), kCountTimeoutSeconds, unused);
                } catch (...) {
                }
                throw;
            }
        }

        metadata.reserve(9);
        metadata.resize(7);
        metadata[1] = part_of(arena, 0, {local_experts}, torch::kInt64);
        metadata[2] = part_of(arena, at_offsets, {local_experts + 1}, torch::kInt64);
        metadata[3] = part_of(arena, at_dst, {tokens, 1}, torch::kInt64);
        metadata[4] = part_of(arena, at_send, {1}, torch::kInt64);
        metadata[5] = part_of(arena, at_snapshot, {tokens, topk}, torch::kInt64);
        metadata[6] = part_of(arena, at_prefix, {1}, torch::kInt64);
        if (expand)  // private eighth entry: slot[t,k] in one lookup
            metadata.push_back(part_of(arena, 2 * count64 + at_table, {tokens, topk}, torch::kInt32));

        int64_t counts[NANOEP_HOST_COUNT_WORDS] = {0, 0, 0, 0};
        const int status = turn.wait(comm.stream(), kCountTimeoutSeconds, counts);
        if (status == NANOEP_ERR_ROUTING) {
            TORCH_CHECK(false, "dispatch routing ids must be -1 or distinct expert ids in [0, ", local_experts, ")",
                        (counts[3] & NANOEP_ROUTING_BAD_EXPERT) ? "; found an id out of range" : "",
                        (counts[3] & NANOEP_ROUTING_DUPLICATE) ? "; found a duplicate expert within a token" : "");
        }
        recv_count = counts[0];
        expanded_capacity = counts[1];
        TORCH_CHECK(recv_count >= 0 && recv_count <= tokens, "dispatch receive count exceeds the source token count");
        TORCH_CHECK(!expand || expanded_capacity <= std::numeric_limits<int32_t>::max(),
                    "expanded capacity exceeds int32 metadata range");
        metadata[0] = part_of(arena, 2 * count64, {recv_count, topk + 2}, torch::kInt32);
        if (ordered) {
            // private ninth entry: assignments in window-wise slot order (replays walk the A assignments only)
            TORCH_CHECK(counts[2] >= 0 && counts[2] <= order_entries, "assignment count exceeds the slot-order list");
            metadata.push_back(part_of(arena, at_order, {counts[2]}, torch::kInt64));
            runtime.note_valid_share(counts[2], tokens * topk);
        }
        const int64_t used_rows = expand ? expanded_capacity : recv_count;
        const bool bound_is_close = used_rows * 5 >= row_bound * 4;  // the bound holds at most 1.25 x the rows in use
        TORCH_CHECK(used_rows <= row_bound, "receive rows exceed their upper bound");
        // the early outputs are kept when every row in use has a place in them and they hold at most 1.25 x those rows
        const bool early_outputs_fit = speculative && used_rows <= early_rows && used_rows * 5 >= early_rows * 4;
        runtime.note_used_rows(geometry, used_rows);
        if (early_outputs_fit) {
            out_x = part_of(out_x, 0, {used_rows, hidden}, torch::kBFloat16);
            if (!expand)
                out_indices = part_of(out_indices, 0, {recv_count, topk}, torch::kInt64);
            if (weights.has_value())
                out_weights = expand ? part_of(out_weights, 0, {used_rows}, torch::kFloat32) : part_of(out_weights, 0, {recv_count, topk}, torch::kFloat32);
        } else {
            // the kernel that writes early outputs that gave way to exact ones may still be running
            if (speculative && marker) {
                marker->discard_written();
                marker->writes(arena);
            }
            allocate_outputs(used_rows, recv_count);
            if (recv_count > 0) {
                if (borrows)
                    wait_on(comm, compute);
                launch_permute(view_of(metadata), recv_count, expanded_capacity);
            }
        }
        if (tokens > 0 && bound_rule)
            runtime.note_output_fill(bound_is_close);
        if (expand)
            runtime.remember_private(metadata, alignment);
    }

    // absent ones at this boundary, made off the path to the launch
    if (expand)
        out_indices = new_tensor({0}, torch::kInt64, here);
    if (!weights.has_value())
        out_weights = new_tensor({0}, torch::kFloat32, here);
    std::vector<torch::Tensor> outputs{out_x, out_indices, out_weights};
    if (async_op) {
        marker->record(compute);
    } else if (marker) {
        wait_on(compute, comm);
        marker->settle();
    }
    return std::make_tuple(std::move(outputs), std::move(metadata), std::array<int64_t, 2>{recv_count, expanded_capacity},
                           async_op ? marker : nullptr);
}

using CombineResult = std::tuple<std::vector<torch::Tensor>, std::shared_ptr<CompletionEvent>>;

CombineResult combine(PeerRuntime& runtime,
                      const torch::Tensor& x,
                      const std::vector<torch::Tensor>& metadata,
                      const c10::optional<torch::Tensor>& weights,
                      const c10::optional<torch::Tensor>& bias,
                      int64_t max_tokens,
                      bool expand,
                      bool allow_multiple_reduction,
                      int num_sms,
                      int64_t comm_stream,
                      int64_t previous_event,
                      bool async_op) {
    TORCH_CHECK(metadata.size() >= 7 && metadata.size() <= 9 && x.defined() && x.dim() == 2 && metadata[5].dim() == 2,
                "combine requires a 2D payload and seven prepared metadata tensors");
    runtime.require_usable();
    const auto device = static_cast<c10::DeviceIndex>(runtime.device());
    DeviceGuard device_guard(device);
    const c10::Device here(c10::DeviceType::CUDA, device);
    TORCH_CHECK(x.is_cuda() && x.device() == here && x.is_contiguous() && x.size(1) > 0,
                "combine x must be contiguous CUDA [N,H] or [C,H] on the runtime device");
    require(x, here, torch::kBFloat16, {-1, -1}, "combine x must be bfloat16");
    TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0, "combine x data pointer must be 16-byte aligned");
    TORCH_CHECK(x.size(1) % kHiddenAlignment == 0, "combine hidden must be a positive multiple of 256");
    TORCH_CHECK(metadata[1].dim() == 1 && metadata[1].numel() > 0,
                "combine metadata requires a [T,K] source snapshot and [L] expert counts");

    const int64_t recv_count = metadata[0].dim() == 2 ? metadata[0].size(0) : -1;
    const int64_t source_tokens = metadata[5].size(0);
    const int64_t hidden = x.size(1);
    const int64_t topk = metadata[5].size(1);
    const int64_t local_experts = metadata[1].numel();
    TORCH_CHECK(topk > 0 && topk <= 32 && topk <= local_experts && source_tokens <= max_tokens && recv_count <= max_tokens,
                "combine routing geometry exceeds expert/token capacity");
    require_handle_tensors(metadata, here, source_tokens, topk, local_experts);
    TORCH_CHECK(expand ? (x.size(0) >= recv_count && (recv_count != 0 || x.size(0) == 0)) : x.size(0) == recv_count,
                "combine x rows do not match the receive layout");
    if (weights.has_value())
        TORCH_CHECK(expand ? describes(*weights, here, torch::kFloat32, {x.size(0)}) : describes(*weights, here, torch::kFloat32, {recv_count, topk}),
                    "combine weights must be contiguous CUDA float32 [N,K] or expanded [C] on the x device");
    if (bias.has_value())
        require(*bias, here, torch::kBFloat16, {source_tokens, hidden},
                "combine bias must be contiguous [T,H], with the output dtype on the x device");
    const int cu_budget = resolve_cu_budget(num_sms, device);

    const auto compute = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device);
    const auto comm = work_stream(comm_stream, compute, device, async_op, cu_budget != 0);
    const StreamSwitch on_comm(comm, compute);
    // (as in dispatch)
    const auto marker = async_op || !same_queue(comm, compute) ? std::make_shared<CompletionEvent>(comm) : nullptr;
    if (marker) {
        marker->reads(metadata);
        marker->reads(x);
        if (weights.has_value())
            marker->reads(*weights);
        if (bias.has_value())
            marker->reads(*bias);
    }

    torch::Tensor combined_x, combined_weights;
    {
        // (as in dispatch: the caller's pool, unless the call is ordered behind an event of its own only, and
        // the order made behind the allocation)
        const StreamSwitch pool(!async_op || previous_event == -1 ? compute : comm, comm);
        combined_x = new_tensor({source_tokens, hidden}, torch::kBFloat16, here);
        if (weights.has_value())
            combined_weights = new_tensor({source_tokens, topk}, torch::kFloat32, here);
        if (marker) {
            marker->writes(combined_x);
            marker->writes(combined_weights);
        }
    }
    order_comm_after_inputs(comm, compute, previous_event, async_op);
    if (source_tokens > 0) {
        // a seven-tensor handle of the latest fresh dispatch gets its slot table back from the runtime
        std::vector<torch::Tensor> handle;
        if (expand && metadata.size() == 7 && tuning_switch("RECALL_ORDER") != 0) {
            handle = metadata;
            runtime.recall_private(handle, -1);
        }
        const auto& lookup = handle.size() > 7 ? handle : metadata;
        const int32_t* table = slot_table(lookup, source_tokens, topk, expand);
        // ... or the table a replayed dispatch of this handle had rebuilt
        std::shared_ptr<PeerRuntime::RebuiltHandle> rebuilt;
        if (table == nullptr && expand && metadata.size() == 7 && recv_count > 0 && tuning_switch("REBUILD_ORDER") != 0) {
            if (!capturing(comm) && (rebuilt = runtime.find_rebuilt(metadata, x.size(0)))) {
                if (rebuilt->made_on != comm.stream()) {
                    if (!rebuilt->ready.query())
                        comm.unwrap().wait(rebuilt->ready);
                    rebuilt->order.record_stream(comm.unwrap());
                }
                table = rebuilt->table.data_ptr<int32_t>();
            }
        }
        check_status(nanoep_combine(x.data_ptr(), weights.has_value() ? weights->data_ptr<float>() : nullptr,
                                    bias.has_value() ? bias->data_ptr() : nullptr, metadata[0].data_ptr<int32_t>(),
                                    metadata[3].data_ptr<int64_t>(), table, recv_count,
                                    x.size(0), source_tokens, static_cast<int>(hidden),
                                    static_cast<int>(topk), expand ? 1 : 0, allow_multiple_reduction ? 1 : 0, combined_x.data_ptr(),
                                    weights.has_value() ? combined_weights.data_ptr<float>() : nullptr, cu_budget, comm.stream()),
                     "combine");
    }

    if (!weights.has_value())
        combined_weights = new_tensor({0}, torch::kFloat32, here);
    std::vector<torch::Tensor> outputs{combined_x, combined_weights};
    if (async_op) {
        marker->record(compute);
    } else if (marker) {
        wait_on(compute, comm);
        marker->settle();
    }
    return std::make_tuple(std::move(outputs), async_op ? marker : nullptr);
}

std::vector<int64_t> window_layout(int ranks, int64_t tokens, int hidden, int topk, int64_t num_experts, bool allow_multiple_reduction) {
    int64_t out[5] = {0, 0, 0, 0, 0};
    const int status = nanoep_window_layout(ranks, tokens, hidden, topk, num_experts, allow_multiple_reduction ? 1 : 0, out);
    if (status != NANOEP_OK)
        throw py::value_error("window_layout requires ranks/topk in [1,32], positive capacity/hidden and num_experts divisible by ranks");
    return {out[0], out[1], out[2], out[3], out[4]};
}

}  // namespace nanoep

// The module's dispatch and combine as plain CPython functions.  A call whose arguments are all positional and of the types
// that the operators take is unpacked here; any other call (keywords, defaults, other types) goes to the bound functions
// below, which say what is wrong with it.  Results and exceptions are theirs.  A small batch's pass is bound by the host, and the
// binding was a part of that: bound -> these, dispatch and combine, the fastest of sixty blocks of passes, ten processes of each (a process
// is in one of two modes): 16 x 256 top-2 replay 14.1 -> 13.7 us (the faster mode 13.3 -> 12.8), 256 x 4096 top-8 14.5 -> 13.9 (13.3 -> 12.8), fresh 21.7 ->
// 21.0 (19.6 -> 19.0) and 22.5 -> 22.1 (21.0 -> 20.5), asynchronous 39.3 -> 39.0 (36.1 -> 35.5).
namespace nanoep {
namespace {

PyObject* g_bound_dispatch = nullptr;
PyObject* g_bound_combine = nullptr;

// What a call's arguments are read into; `fits` turns false at the first that is not what the operator takes.
class Arguments {
   public:
    explicit Arguments(PyObject* const* args) : next_(args) {}
    bool fits() const { return fits_; }

    PeerRuntime* runtime() {
        const py::handle object(*next_++);
        if (py::isinstance<PeerRuntime>(object))
            return object.cast<PeerRuntime*>();
        fits_ = false;
        return nullptr;
    }
    torch::Tensor tensor() {
        PyObject* object = *next_++;
        if (THPVariable_Check(object))
            return THPVariable_Unpack(object);
        fits_ = false;
        return {};
    }
    c10::optional<torch::Tensor> tensor_or_none() {
        if (*next_ == Py_None) {
            ++next_;
            return c10::nullopt;
        }
        return tensor();
    }
    std::vector<torch::Tensor> tensors() {
        std::vector<torch::Tensor> all;
        PyObject* list = *next_++;
        if (!PyList_CheckExact(list)) {
            fits_ = false;
            return all;
        }
        const Py_ssize_t count = PyList_GET_SIZE(list);
        all.reserve(static_cast<size_t>(count));
        for (Py_ssize_t i = 0; i < count; ++i) {
            PyObject* object = PyList_GET_ITEM(list, i);
            if (!THPVariable_Check(object)) {
                fits_ = false;
                return all;
            }
            all.push_back(THPVariable_Unpack(object));
        }
        return all;
    }
    int64_t integer() {
        PyObject* object = *next_++;
        int overflow = 1;
        const long long value = PyLong_CheckExact(object) ? PyLong_AsLongLongAndOverflow(object, &overflow) : 0;
        fits_ = fits_ && overflow == 0;
        return value;
    }
    int small_integer() {
        const int64_t value = integer();
        fits_ = fits_ && value >= std::numeric_limits<int>::min() && value <= std::numeric_limits<int>::max();
        return static_cast<int>(value);
    }
    bool boolean() {
        PyObject* object = *next_++;
        fits_ = fits_ && PyBool_Check(object);
        return object == Py_True;
    }

   private:
    PyObject* const* next_;
    bool fits_ = true;
};

py::list wrapped(std::vector<torch::Tensor>& tensors) {
    py::list list(tensors.size());
    for (size_t i = 0; i < tensors.size(); ++i) {
        PyObject* object = THPVariable_Wrap(std::move(tensors[i]));
        if (object == nullptr)
            throw py::error_already_set();
        PyList_SET_ITEM(list.ptr(), static_cast<Py_ssize_t>(i), object);
    }
    return list;
}

py::object wrapped(const std::shared_ptr<CompletionEvent>& event) { return event ? py::cast(event) : py::none(); }

PyObject* g_rethrow = nullptr;                  // a bound function that throws this thread's exception
thread_local std::exception_ptr g_exception;

// Runs `call`; the binding makes its exceptions Python's, as it does those of the bound functions.  A thread that is ended inside
// the call unwinds on.
template <class Call>
PyObject* guarded(const Call& call) {
    try {
        return call();
    } catch (abi::__forced_unwind&) {
        throw;
    } catch (...) {
        g_exception = std::current_exception();
    }
    return PyObject_CallNoArgs(g_rethrow);
}

constexpr Py_ssize_t kDispatchArguments = 16, kCombineArguments = 12;

PyObject* call_dispatch(PyObject*, PyObject* const* args, Py_ssize_t count, PyObject* names) {
    if (count != kDispatchArguments || names != nullptr)
        return PyObject_Vectorcall(g_bound_dispatch, args, static_cast<size_t>(count), names);
    return guarded([&]() -> PyObject* {
        Arguments from(args);
        PeerRuntime* runtime = from.runtime();
        const torch::Tensor x = from.tensor(), indices = from.tensor();
        const auto weights = from.tensor_or_none();
        const int64_t experts = from.integer(), max_tokens = from.integer(), alignment = from.integer();
        const auto cached = from.tensors();
        const int64_t cached_capacity = from.integer();
        const bool multiple_reduction = from.boolean(), expand = from.boolean(), zero_padding = from.boolean();
        const int num_sms = from.small_integer();
        const int64_t comm_stream = from.integer(), previous_event = from.integer();
        const bool async_op = from.boolean();
        if (!from.fits())
            return PyObject_Vectorcall(g_bound_dispatch, args, static_cast<size_t>(count), names);
        DispatchResult result;
        {
            py::gil_scoped_release without_interpreter;
            result = dispatch(*runtime, x, indices, weights, experts, max_tokens, alignment, cached, cached_capacity, multiple_reduction, expand,
                              zero_padding, num_sms, comm_stream, previous_event, async_op);
        }
        py::list counts(2);
        counts[0] = py::int_(std::get<2>(result)[0]);
        counts[1] = py::int_(std::get<2>(result)[1]);
        return py::make_tuple(wrapped(std::get<0>(result)), wrapped(std::get<1>(result)), counts, wrapped(std::get<3>(result))).release().ptr();
    });
}

PyObject* call_combine(PyObject*, PyObject* const* args, Py_ssize_t count, PyObject* names) {
    if (count != kCombineArguments || names != nullptr)
        return PyObject_Vectorcall(g_bound_combine, args, static_cast<size_t>(count), names);
    return guarded([&]() -> PyObject* {
        Arguments from(args);
        PeerRuntime* runtime = from.runtime();
        const torch::Tensor x = from.tensor();
        const auto metadata = from.tensors();
        const auto weights = from.tensor_or_none(), bias = from.tensor_or_none();
        const int64_t max_tokens = from.integer();
        const bool expand = from.boolean(), multiple_reduction = from.boolean();
        const int num_sms = from.small_integer();
        const int64_t comm_stream = from.integer(), previous_event = from.integer();
        const bool async_op = from.boolean();
        if (!from.fits())
            return PyObject_Vectorcall(g_bound_combine, args, static_cast<size_t>(count), names);
        CombineResult result;
        {
            py::gil_scoped_release without_interpreter;
            result = combine(*runtime, x, metadata, weights, bias, max_tokens, expand, multiple_reduction, num_sms, comm_stream, previous_event,
                             async_op);
        }
        return py::make_tuple(wrapped(std::get<0>(result)), wrapped(std::get<1>(result))).release().ptr();
    });
}

// Puts `call` in the place of the module's bound function of that name, with its docstring, and keeps that one for the calls it
// passes on.
struct CallAhead {
    PyMethodDef definition;
    std::string doc;
};

template <class Function>
void call_ahead_of(py::module_& module, CallAhead& ahead, const char* name, Function call, PyObject*& bound) {
    const py::object function = module.attr(name);
    ahead.doc = py::str(function.attr("__doc__"));
    bound = py::object(function).release().ptr();
    ahead.definition = {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call)), METH_FASTCALL | METH_KEYWORDS, ahead.doc.c_str()};
    module.attr(name) = py::reinterpret_steal<py::object>(PyCFunction_NewEx(&ahead.definition, nullptr, module.attr("__name__").ptr()));
}

}  // namespace
}  // namespace nanoep

PYBIND11_MODULE(TORCH_EXTENSION_NAME, module) {
    module.doc() = "MI355X dispatch / combine host extension (ahead-of-time HIP kernels behind a C ABI)";
    module.attr("abi_version") = nanoep_abi_version();
    // Kernels are compiled ahead of time: the JIT warm-up entry points are accepted and ignored.
    module.def("init_jit", [](const std::string&) {});
    module.def("prepare_dispatch", [](py::args, py::kwargs) {});
    module.def("prepare_combine", [](py::args, py::kwargs) {});
    module.def("dispatch", &nanoep::dispatch, py::arg("runtime"), py::arg("x"), py::arg("indices"), py::arg("weights"),
               py::arg("num_experts"), py::arg("max_tokens"), py::arg("alignment"), py::arg("cached_metadata"),
               py::arg("cached_expanded_capacity"), py::arg("allow_multiple_reduction"), py::arg("expand"), py::arg("zero_padding"),
               py::arg("num_sms"), py::arg("comm_stream"), py::arg("previous_event") = -1, py::arg("async_op") = true,
               py::call_guard<py::gil_scoped_release>());
    module.def("combine", &nanoep::combine, py::arg("runtime"), py::arg("x"), py::arg("metadata"), py::arg("weights"), py::arg("bias"),
               py::arg("max_tokens"), py::arg("expand"), py::arg("allow_multiple_reduction"), py::arg("num_sms"), py::arg("comm_stream"),
               py::arg("previous_event") = -1, py::arg("async_op") = true, py::call_guard<py::gil_scoped_release>());
    module.def("window_layout", &nanoep::window_layout, py::arg("ranks"), py::arg("tokens"), py::arg("hidden"), py::arg("topk"),
               py::arg("num_experts"), py::arg("allow_multiple_reduction") = false);
    py::class_<nanoep::PeerRuntime>(module, "PeerRuntime")
        .def(py::init<int, int, int64_t>())
        .def("export_local_handle", &nanoep::PeerRuntime::export_local_handle)
        .def("import_peer_handles", &nanoep::PeerRuntime::import_peer_handles)
        .def("peer_addresses", &nanoep::PeerRuntime::peer_addresses)
        .def("local_window", &nanoep::PeerRuntime::local_window)
        .def("barrier", &nanoep::PeerRuntime::barrier)
        .def("barrier", &nanoep::PeerRuntime::barrier_at)
        .def("close_peer_mappings", &nanoep::PeerRuntime::close_peer_mappings)
        .def("private_recalls", &nanoep::PeerRuntime::private_recalls)
        .def("rebuilds", &nanoep::PeerRuntime::rebuilds)
        .def("budget_stream", &nanoep::PeerRuntime::budget_stream)
        .def("budget_stream_cus", &nanoep::PeerRuntime::budget_stream_cus)
        .def("counts_failed", &nanoep::PeerRuntime::counts_failed)
        .def("prefers_exact_outputs", &nanoep::PeerRuntime::prefers_exact_outputs)
        .def("valid_share_65536", &nanoep::PeerRuntime::valid_share_65536)
        .def("lose_counts_for_test", &nanoep::PeerRuntime::lose_counts_for_test)
        .def("close", &nanoep::PeerRuntime::close);
    py::class_<nanoep::CompletionEvent, std::shared_ptr<nanoep::CompletionEvent>>(module, "CompletionEvent")
        .def("current_stream_wait", &nanoep::CompletionEvent::current_stream_wait);
    static nanoep::CallAhead dispatch_ahead, combine_ahead;
    nanoep::call_ahead_of(module, dispatch_ahead, "dispatch", &nanoep::call_dispatch, nanoep::g_bound_dispatch);
    nanoep::call_ahead_of(module, combine_ahead, "combine", &nanoep::call_combine, nanoep::g_bound_combine);
    nanoep::g_rethrow = py::cpp_function([] { std::rethrow_exception(std::exchange(nanoep::g_exception, nullptr)); }).release().ptr();
}
