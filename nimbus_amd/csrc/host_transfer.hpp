// Copies between host arrays and the device through a ring of pinned slots.
//
// A pageable copy by the runtime moves 10 GB/s into freshly mapped memory (18
// into warm): one thread copies and takes the page faults, and nothing
// overlaps it. Here the device side of chunk c (a kernel that reads or writes
// its slot over the host link, 49-53 GB/s) runs while a few threads move other
// chunks between slots and the caller's arrays (29 GB/s per thread in warm
// pages, 13 in fresh ones, 55 together). Small calls, and memory of the runtime
// (pinned, or a device's), take other ways: see copy() and place().
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace nimbus
{

// A whole array and its copy on the device. No bytes: no copy.
struct ArrayCopy
{
    void* dev;
    void* host;
    std::size_t bytes;
};

// How the device side of a transfer gets at one of the caller's arrays.
enum class Reach
{
    Host,     // ordinary memory: std::memcpy to or from a slot
    Runtime,  // memory of the runtime that a kernel here may not touch: hipMemcpy to or from a slot
    Kernel    // a kernel on the context's device reads or writes the array itself
};

// A contiguous piece of one of the caller's arrays.
struct HostChunk
{
    char* host;
    std::size_t bytes;
    Reach reach;
};

class HostTransfer
{
public:
    static constexpr std::size_t kSlot = std::size_t(2) << 20;
    static constexpr int kSlots = 10;
    static constexpr int kThreads = 6;
    // Bytes for each thread that copies, fields turned by the kernel and whole
    // arrays. Starting a thread, and the release of device memory beside it, cost
    // what it saves on less: fields with 1 MB against 4 MB for each, us: 9 of
    // 64 x 64 x 48 doubles 435 to 408, the acoustic contract of 84 x 90 x 60 cells
    // 2,216 to 1,815 (2 MB 1,965). Arrays with 1, 2 and 4 MB: the transport
    // contract of 96 x 100 x 70 cells 2,680, 2,460 and 2,540, of 118 x 122 x 60
    // 3,110, 3,130 and 3,640.
    static constexpr std::size_t kFieldShare = std::size_t(4) << 20;
    static constexpr std::size_t kArrayShare = std::size_t(2) << 20;
    // Whole arrays take the ring from these sizes of one direction on (down:
    // and of an array on average). Below them the ring's threads and the copy,
    // event and wait of every chunk cost more than they overlap. Plain copies
    // against the ring, us: down (18 GB/s plain), 16 x 128 KB 246 to 297, 4 x 512 KB
    // 116 to 133, 8 x 512 KB 258 to 225, 2 x 2 MB 230 to 180, 4 x 2 MB 461 to 318; up,
    // where a plain copy reads warm pages at 35 GB/s and runs beside the caller's
    // next allocation, whole calls with 9 arrays of 96 x 96 x 60 floats (20 MB)
    // 1,850 to 2,120, of 112 x 112 x 60 (27 MB) 2,500 to 2,900, with 4 of
    // 160 x 160 x 80 (33 MB) 3,840 to 3,530, with 5 of them 6,590 to 6,040.
    static constexpr std::size_t kRingDown = std::size_t(4) << 20;
    static constexpr std::size_t kRingArray = std::size_t(512) << 10;
    static constexpr std::size_t kRingUp = std::size_t(28) << 20;
    // Whether `count` arrays of `bytes` together take the ring.
    static constexpr bool takes_ring(bool up, std::size_t bytes, std::size_t count)
    {
        return up ? bytes >= kRingUp : bytes >= kRingDown && bytes >= count * kRingArray;
    }

    HostTransfer() = default;
    HostTransfer(const HostTransfer&) = delete;
    HostTransfer& operator=(const HostTransfer&) = delete;
    ~HostTransfer()
    {
        for (hipEvent_t e : events_) hipEventDestroy(e);
        if (slots_) hipHostFree(slots_);
    }

    // Moves the chunks to (up) or from the device; launch(c, p) enqueues the
    // device side of chunk c on `stream` against p, its slot or (Reach::Kernel) its
    // array. Returns when the caller's arrays are read or written. Transfers of
    // one ring run one after the other.
    template <class Launch>
    hipError_t run(int device, hipStream_t stream, bool up, const std::vector<HostChunk>& chunks, Launch launch,
                   std::size_t share = kFieldShare)
    {
        std::lock_guard<std::mutex> one(busy_);
        State st;
        st.n = int(chunks.size());
        st.copied.assign(chunks.size(), 0);
        std::size_t bytes = 0, copies = 0;
        for (const HostChunk& c : chunks)
            if (c.reach != Reach::Kernel)
            {
                bytes += c.bytes;
                ++copies;
            }
        hipError_t e = prepare(copies != 0);
        if (e != hipSuccess) return e;
        const std::size_t most = !up && shared(chunks) ? 1 : std::min(std::size_t(kThreads), copies);
        const int want = int(std::min(most, (bytes + share / 2) / share));
        std::vector<std::thread> team;
        team.reserve(kThreads);  // no allocation once a thread runs
        try
        {
            for (int t = 1; t < want; ++t)
                team.emplace_back([&] {
                    hipSetDevice(device);
                    std::unique_lock<std::mutex> lock(st.m);
                    while (true)
                    {
                        st.cv.wait(lock, [&] { return st.over() || st.can_copy(up); });
                        if (st.over()) return;
                        copy(st, lock, chunks, up);
                    }
                });
        }
        catch (const std::exception&)
        {
            // no thread, or no memory for its state: those that did start, and this one, do the work
        }
        {
            std::unique_lock<std::mutex> lock(st.m);
            while (st.issued < st.n && st.error == hipSuccess)
            {
                const int c = st.issued;
                if (up ? st.copied[c] : c < kSlots || st.copied[c - kSlots])
                {
                    lock.unlock();
                    hipError_t r = launch(c, chunks[c].reach == Reach::Kernel ? chunks[c].host : slot(c));
                    if (r == hipSuccess) r = hipEventRecord(events_[c % kSlots], stream);
                    lock.lock();
                    if (r != hipSuccess) st.error = r;
                    else ++st.issued;
                    st.cv.notify_all();
                }
                else if (!st.over() && st.can_copy(up)) copy(st, lock, chunks, up);
                else st.cv.wait(lock);
            }
            while (!st.over())
                if (st.can_copy(up)) copy(st, lock, chunks, up);
                else st.cv.wait(lock);
        }
        for (std::thread& t : team) t.join();
        e = hipStreamSynchronize(stream);
        return st.error != hipSuccess ? st.error : e;
    }

    // Copies whole arrays to (up) or from the device. Downloads are complete on
    // return; uploads precede what is enqueued on `stream` next, and the arrays
    // are read by the time that `stream` has run.
    hipError_t copy(int device, hipStream_t stream, bool up, std::vector<ArrayCopy> arrays)
    {
        auto rings = [up](auto first, auto last) {
            std::size_t bytes = 0, count = 0;
            for (; first != last; ++first)
            {
                bytes += first->bytes;
                count += first->bytes != 0;
            }
            return takes_ring(up, bytes, count);
        };
        // first what is copied plainly: everything below the ring's sizes, and memory
        // of the runtime, pinned or any device's, which its copies move without a slot
        auto staged = arrays.end();
        if (rings(arrays.begin(), arrays.end()))
        {
            staged = std::stable_partition(arrays.begin(), arrays.end(), [&](const ArrayCopy& a) {
                return a.bytes == 0 || of_runtime(a.host);
            });
            if (!rings(staged, arrays.end())) staged = arrays.end();
        }
        for (auto a = arrays.begin(); a != staged; ++a)
        {
            if (a->bytes == 0) continue;
            const hipError_t e = hipMemcpyAsync(up ? a->dev : a->host, up ? a->host : a->dev, a->bytes,
                                                hipMemcpyDefault, stream);
            if (e != hipSuccess) return e;
        }
        if (staged == arrays.end()) return up ? hipSuccess : hipStreamSynchronize(stream);
        std::vector<HostChunk> chunks;
        std::vector<char*> dev;
        for (auto a = staged; a != arrays.end(); ++a)
            for (std::size_t o = 0; o < a->bytes; o += kSlot)
            {
                chunks.push_back(HostChunk{static_cast<char*>(a->host) + o, std::min(kSlot, a->bytes - o), Reach::Host});
                dev.push_back(static_cast<char*>(a->dev) + o);
            }
        return run(device, stream, up, chunks, [&](int c, char* p) {
            return hipMemcpyAsync(up ? dev[c] : p, up ? p : dev[c], chunks[c].bytes, hipMemcpyDefault, stream);
        }, kArrayShare);
    }

    // How a kernel on `device` reaches a caller's array of elements of `size`
    // bytes, and at which address: memory of its own device and host memory
    // pinned for it, aligned and allocated over the whole array.
    struct Place
    {
        Reach reach;
        char* at;
    };
    static Place place(int device, const void* p, std::size_t bytes, std::size_t size)
    {
        hipPointerAttribute_t at{};
        Place r{Reach::Host, static_cast<char*>(const_cast<void*>(p))};
        if (!of_runtime(p, &at)) return r;
        if (at.type != hipMemoryTypeHost) r.reach = Reach::Runtime;
        char* const q = static_cast<char*>(at.type == hipMemoryTypeHost ? at.devicePointer : r.at);
        if (!q || (at.type != hipMemoryTypeHost && at.type != hipMemoryTypeDevice) || at.device != device ||
            reinterpret_cast<std::uintptr_t>(q) % size != 0)
            return r;
        hipDeviceptr_t base = nullptr;
        std::size_t n = 0;
        if (hipMemGetAddressRange(&base, &n, q) == hipSuccess)
        {
            const std::size_t o = std::size_t(q - static_cast<char*>(base));
            if (o <= n && bytes <= n - o) return Place{Reach::Kernel, q};
        }
        hipGetLastError();
        return r;
    }

    // Whether the runtime knows an array's memory (pinned, or any device's).
    static bool of_runtime(const void* p, hipPointerAttribute_t* at = nullptr)
    {
        hipPointerAttribute_t own{};
        if (!at) at = &own;
        const bool known = hipPointerGetAttributes(at, p) == hipSuccess && at->type != hipMemoryTypeUnregistered;
        hipGetLastError();  // an ordinary host array is no error
        return known;
    }

private:
    struct State
    {
        std::mutex m;
        std::condition_variable cv;
        int n = 0, issued = 0, next = 0;  // chunks; whose device side is enqueued; whose copy is taken
        std::vector<char> copied;
        hipError_t error = hipSuccess;
        bool over() const { return next >= n || error != hipSuccess; }
        // chunk `next` has its data in the slot (down), or the slot's last user is enqueued (up)
        bool can_copy(bool up) const { return up ? next < issued + kSlots : next < issued; }
    };

    // Whether two of the caller's arrays share memory: downloads to them go in order.
    static bool shared(const std::vector<HostChunk>& chunks)
    {
        std::vector<std::pair<char*, char*>> arrays;
        for (const HostChunk& c : chunks)
            if (!arrays.empty() && arrays.back().second == c.host) arrays.back().second += c.bytes;
            else arrays.emplace_back(c.host, c.host + c.bytes);
        std::sort(arrays.begin(), arrays.end());
        for (std::size_t q = 1; q < arrays.size(); ++q)
            if (arrays[q].first < arrays[q - 1].second) return true;
        return false;
    }

    char* slot(int c) const { return static_cast<char*>(slots_) + std::size_t(c % kSlots) * kSlot; }

    // Takes the next chunk and copies it, unlocked meanwhile.
    void copy(State& st, std::unique_lock<std::mutex>& lock, const std::vector<HostChunk>& chunks, bool up)
    {
        const int c = st.next++;
        lock.unlock();
        hipError_t r = hipSuccess;
        if (!up || c >= kSlots) r = hipEventSynchronize(events_[c % kSlots]);
        const HostChunk& k = chunks[c];
        if (r == hipSuccess && k.reach != Reach::Kernel)
        {
            void* const to = up ? slot(c) : k.host;
            const void* const from = up ? k.host : slot(c);
            if (k.reach == Reach::Runtime) r = hipMemcpy(to, from, k.bytes, hipMemcpyDefault);
            else std::memcpy(to, from, k.bytes);
        }
        lock.lock();
        if (r != hipSuccess) st.error = r;
        st.copied[c] = 1;
        st.cv.notify_all();
    }

    hipError_t prepare(bool slots)
    {
        while (int(events_.size()) < kSlots)
        {
            hipEvent_t ev = nullptr;
            const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
            if (e != hipSuccess) return e;
            events_.push_back(ev);
        }
        if (slots_ || !slots) return hipSuccess;
        // coherent, whatever HIP_HOST_COHERENT says: a slot is read once its event has passed,
        // which makes no other memory visible to the host
        const hipError_t e = hipHostMalloc(&slots_, kSlot * kSlots, hipHostMallocCoherent);
        if (e != hipSuccess) slots_ = nullptr;
        return e;
    }

    std::mutex busy_;
    void* slots_ = nullptr;
    std::vector<hipEvent_t> events_;
};

}  // namespace nimbus
