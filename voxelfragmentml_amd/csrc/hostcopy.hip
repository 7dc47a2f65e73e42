// Device memory to pageable host memory.  The runtime's copy stages through pinned memory with one host thread: 17.9 GB/s,
// where the link carries 57.  Here chunks are written to a ring of pinned slots by kernels, and the calling thread and
// a few helpers copy filled slots on to the caller's memory while the device fills the next: 44 GB/s for 32 MiB.
#include "hostcopy.hpp"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace vf {

namespace {

constexpr uint32_t kChunk = 1u << 19;        // bytes of a slot
constexpr uint32_t kSlots = 16;              // 8 MiB of pinned memory
constexpr uint32_t kGroup = 4;               // chunks of one launch
constexpr uint32_t kStageThreads = 256;
constexpr uint32_t kStagePart = 1u << 15;    // bytes of a workgroup
constexpr uint32_t kStageBlocks = kChunk / kStagePart;
constexpr uint32_t kHelpers = 3;
constexpr size_t kStagedMin = 1u << 20;      // fewer bytes: the runtime's copy (512 KiB take it 30 us, this one 33; 1.7 MiB 97 and 75)
// Bytes an object has to copy before it makes a pool (one that is there is used from kStagedMin on): making and dropping it takes
// 120 to 150 us, and a MiB by it 33 us less than by the runtime.  A program that makes a grid, reads it and drops it took 427 us
// for one of 82^3 cells with a pool each time, 323 without.
constexpr size_t kPoolPays = 4u << 20;

// Chunk blockIdx.y: bytes of src to dst, equally aligned; workgroup b's flag is set to seq when its part is in host
// memory.  A launch takes kGroup chunks: the gap between two launches and the wait for the last store of one cost 7 us,
// as much as the link takes for 400 KB.
struct StageArgs {
    struct {
        const uint8_t* src;
        uint8_t* dst;
        uint32_t* flags;
        uint32_t bytes, seq;
    } c[kGroup];
};
__global__ __launch_bounds__(kStageThreads) void k_stage(StageArgs a)
{
    const uint8_t* src = a.c[blockIdx.y].src;
    uint8_t* dst = a.c[blockIdx.y].dst;
    const uint32_t bytes = a.c[blockIdx.y].bytes, seq = a.c[blockIdx.y].seq;
    uint32_t* flags = a.c[blockIdx.y].flags;
    if (blockIdx.x * kStagePart >= bytes) return;  // a shorter chunk beside longer ones
    const uint32_t head = min(bytes, (uint32_t)(-(uintptr_t)src & 15u));  // up to the first 16-byte boundary
    const uint32_t body = (bytes - head) / 16u;
    const uint4* s = reinterpret_cast<const uint4*>(src + head);
    uint4* d = reinterpret_cast<uint4*>(dst + head);
    constexpr uint32_t kVecs = kStagePart / 16u, kRun = kVecs / kStageThreads;
    uint4 q[kRun];
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t i = blockIdx.x * kVecs + r * kStageThreads + threadIdx.x;
        if (i < body) q[r] = s[i];
    }
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t i = blockIdx.x * kVecs + r * kStageThreads + threadIdx.x;
        if (i < body) d[i] = q[r];
    }
    if (blockIdx.x == 0) {
        if (threadIdx.x < head) dst[threadIdx.x] = src[threadIdx.x];
        const uint32_t tail = head + 16u * body;  // at most 15 bytes after it
        if (threadIdx.x < bytes - tail) dst[tail + threadIdx.x] = src[tail + threadIdx.x];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flags + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

class CopyPool {
public:
    CopyPool()
    {
        VF_HIP(hipHostMalloc(reinterpret_cast<void**>(&base_), kSlots * kSlotBytes + kSlots * kStageBlocks * 4,
                             hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
        flags_ = reinterpret_cast<uint32_t*>(base_ + kSlots * kSlotBytes);
        std::memset(flags_, 0, kSlots * kStageBlocks * 4);
    }
    ~CopyPool()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (std::thread& t : helpers_) t.join();
        if (base_) (void)hipHostFree(base_);
    }
    // false: another thread is using the pool
    bool run(const std::vector<HostCopies::Part>& list, hipStream_t s)
    {
        std::unique_lock<std::mutex> own(busy_, std::try_to_lock);
        if (!own.owns_lock()) return false;
        chunks_.clear();
        for (const HostCopies::Part& p : list)
            for (size_t at = 0; at < p.bytes; at += kChunk)
                chunks_.push_back(Chunk{ p.dst + at, p.src + at, (uint32_t)std::min<size_t>(kChunk, p.bytes - at) });
        const uint32_t n = (uint32_t)chunks_.size();
        for (uint32_t k = 0; k < kSlots; ++k) copied_[k].store(0, std::memory_order_relaxed);
        seq0_ = seq_;
        seq_ += n;
        launched_.store(0, std::memory_order_relaxed);
        failed_.store(false, std::memory_order_relaxed);
        next_.store(0, std::memory_order_relaxed);
        uint32_t queued = 0;
        bool awake = false;
        try {
            const uint32_t helpers = std::min<uint32_t>(kHelpers, n - 1);
            try {
                while (helpers_.size() < helpers) helpers_.emplace_back([this, r = round_] { help(r); });
            } catch (const std::system_error&) {  // no more threads: those there are, or the caller alone
            }
            auto free_slot = [&](uint32_t i) {
                return i < kSlots || copied_[i % kSlots].load(std::memory_order_acquire) == i - kSlots + 1;
            };
            auto queue = [&] {  // the next chunks, when all their slots are free
                while (queued < n) {
                    const uint32_t k = std::min(kGroup, n - queued);
                    StageArgs a;
                    uint32_t most = 0;
                    for (uint32_t j = 0; j < k; ++j) {
                        const uint32_t i = queued + j, slot = i % kSlots;
                        if (!free_slot(i)) return;
                        const Chunk& c = chunks_[i];
                        a.c[j] = { c.src, at(slot, c.src), flags_ + slot * kStageBlocks, c.bytes, seq0_ + i + 1 };
                        most = std::max(most, c.bytes);
                    }
                    k_stage<<<dim3(ceil_div(most, kStagePart), k), kStageThreads, 0, s>>>(a);
                    VF_CHECK_LAUNCH();
                    launched_.store(queued += k, std::memory_order_release);
                }
            };
            HostPause pause;
            for (;;) {
                queue();
                uint32_t i = next_.load(std::memory_order_relaxed);
                if (i >= n) break;
                if (i >= queued) {  // its slot is still being copied by a helper
                    pause();
                    continue;
                }
                if (!filled(i)) {
                    wait(i, s, queue);
                    continue;
                }
                if (!awake && n > 1) {  // helpers are woken when there is something to copy
                    awake = true;
                    {
                        std::lock_guard<std::mutex> lk(mu_);
                        ++round_;
                        open_ = true;
                    }
                    cv_.notify_all();
                }
                if (next_.compare_exchange_strong(i, i + 1)) copy(i);
            }
        } catch (...) {
            failed_.store(true);
            settle(awake);
            (void)hipStreamSynchronize(s);  // kernels already queued still write the slots
            throw;
        }
        settle(awake);
        return true;
    }

private:
    struct Chunk {
        uint8_t* dst;
        const uint8_t* src;
        uint32_t bytes;
    };
    static constexpr size_t kSlotBytes = kChunk + 64;

    uint8_t* at(uint32_t slot, const uint8_t* src) const { return base_ + slot * kSlotBytes + ((uintptr_t)src & 15u); }
    bool filled(uint32_t i) const
    {
        const uint32_t* f = flags_ + (i % kSlots) * kStageBlocks;
        const uint32_t blocks = ceil_div(chunks_[i].bytes, kStagePart);
        for (uint32_t b = 0; b < blocks; ++b)
            if (__atomic_load_n(f + b, __ATOMIC_ACQUIRE) != seq0_ + i + 1) return false;
        return true;
    }
    void copy(uint32_t i)
    {
        const Chunk& c = chunks_[i];
        std::memcpy(c.dst, at(i % kSlots, c.src), c.bytes);
        copied_[i % kSlots].store(i + 1, std::memory_order_release);
    }
    // until chunk i is filled, a helper took it, or the device failed
    template <class F>
    void wait(uint32_t i, hipStream_t s, F&& queue)
    {
        auto since = std::chrono::steady_clock::now();
        HostPause pause;
        while (!filled(i) && next_.load(std::memory_order_relaxed) == i) {
            queue();
            pause();
            if (std::chrono::steady_clock::now() - since > std::chrono::milliseconds(20)) {
                // the work before the copies takes longer, or the device failed
                VF_HIP(hipStreamSynchronize(s));
                if (!filled(i) && next_.load() == i) fail(VF_ERR_DEVICE, "copy to host memory stopped");
                since = std::chrono::steady_clock::now();
            }
        }
    }
    // until no helper looks at the chunks any more: those that have not woken up yet miss the round
    void settle(bool awake)
    {
        if (!awake) return;
        std::unique_lock<std::mutex> lk(mu_);
        open_ = false;
        done_.wait(lk, [&] { return active_ == 0; });
    }
    void help(uint64_t seen)
    {
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return stop_ || (round_ != seen && open_); });
                if (stop_) return;
                seen = round_;
                ++active_;
            }
            const uint32_t n = (uint32_t)chunks_.size();
            HostPause pause;
            for (;;) {
                uint32_t i = next_.load();
                if (i >= n || failed_.load()) break;
                if (i < launched_.load(std::memory_order_acquire) && filled(i)) {
                    if (next_.compare_exchange_strong(i, i + 1)) copy(i);
                } else {
                    pause();
                }
            }
            {
                std::lock_guard<std::mutex> lk(mu_);
                --active_;
            }
            done_.notify_all();
        }
    }

    std::mutex busy_, mu_;
    std::condition_variable cv_, done_;
    std::vector<std::thread> helpers_;
    uint64_t round_ = 0;
    uint32_t active_ = 0;  // helpers in the round
    bool open_ = false;    // helpers may still join it
    bool stop_ = false;
    uint8_t* base_ = nullptr;
    uint32_t* flags_ = nullptr;
    uint32_t seq_ = 0, seq0_ = 0;
    std::vector<Chunk> chunks_;
    std::atomic<uint32_t> next_{ 0 }, launched_{ 0 }, copied_[kSlots] = {};
    std::atomic<bool> failed_{ false };
};

namespace {
// The pool that some object holds; make: or a new one.  None where there is no pinned memory for it.
std::shared_ptr<CopyPool> shared_pool(bool make)
{
    static std::mutex mu;
    static std::weak_ptr<CopyPool> pool;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<CopyPool> p = pool.lock();
    if (!p && make) {
        try {
            p = std::make_shared<CopyPool>();
        } catch (const Exception&) {
            return nullptr;
        }
        pool = p;
    }
    return p;
}

// memory the device copies to at the link's rate by itself: pinned, managed or its own
bool device_reaches(const void* p)
{
    hipPointerAttribute_t a;
    const hipError_t e = hipPointerGetAttributes(&a, p);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess && a.type != hipMemoryTypeUnregistered;
}
}  // namespace

void HostCopies::run(hipStream_t s)
{
    const bool none = list_.empty();
    if (start(s) || none) VF_HIP(hipStreamSynchronize(s));
}

bool HostCopies::start(hipStream_t s)
{
    const std::vector<Part> list = std::move(list_);
    list_.clear();
    size_t total = 0;
    for (const Part& p : list) total += p.bytes;
    std::vector<Part> staged;
    if (total >= kStagedMin)
        for (const Part& p : list)
            if (!device_reaches(p.dst)) staged.push_back(p);
    bool direct = staged.size() < list.size();  // false for an empty list
    if (direct)
        for (const Part& p : list)
            if (staged.empty() || device_reaches(p.dst)) VF_HIP(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s));
    if (!staged.empty()) {
        for (const Part& p : staged) asked_ += p.bytes;
        if (!pool_) pool_ = shared_pool(asked_ >= kPoolPays);
        if (!pool_ || !pool_->run(staged, s)) {  // no pool, or in use by another thread
            direct = true;
            for (const Part& p : staged) VF_HIP(hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s));
        }
    }
    return direct;
}

}  // namespace vf
