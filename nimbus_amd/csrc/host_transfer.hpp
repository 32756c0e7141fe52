// Copies between host arrays and the device through a ring of pinned slots.
//
// A pageable copy by the runtime moves 10 GB/s into freshly mapped memory (18
// into warm): one thread copies and takes the page faults, and nothing
// overlaps it. Here the device side of chunk c (a kernel that reads or writes
// its slot over the host link, 49-53 GB/s) runs while a few threads move other
// chunks between slots and the caller's arrays (29 GB/s per thread in warm
// pages, 13 in fresh ones, 55 together).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
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
    static constexpr std::size_t kRingUp = std::size_t(32) << 20;
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
    hipError_t run(int device, hipStream_t stream, bool up, const std::vector<HostChunk>& chunks, Launch launch)
    {
        std::lock_guard<std::mutex> one(busy_);
        hipError_t e = prepare();
        if (e != hipSuccess) return e;
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
        // a thread for each 4 MB: one for each MB took 2,040 us where this takes 1,910 (a contract
        // call of 13 arrays of 96 x 96 x 60 floats) and 435 where this takes 408 (9 of 64 x 64 x 48
        // doubles), in starting them and in the release of device memory beside them
        const int want = int(std::min<std::size_t>({std::size_t(kThreads), copies, bytes >> 22}));
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
        catch (const std::system_error&)
        {
            // the threads that did start, and this one, do the work
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
    hipError_t copy(int device, hipStream_t stream, bool up, const std::vector<ArrayCopy>& arrays)
    {
        std::size_t bytes = 0, count = 0;
        for (const ArrayCopy& a : arrays)
        {
            bytes += a.bytes;
            count += a.bytes != 0;
        }
        const hipMemcpyKind kind = up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
        if (!takes_ring(up, bytes, count))
        {
            for (const ArrayCopy& a : arrays)
            {
                if (a.bytes == 0) continue;
                const hipError_t e = hipMemcpyAsync(up ? a.dev : a.host, up ? a.host : a.dev, a.bytes, kind, stream);
                if (e != hipSuccess) return e;
            }
            return up ? hipSuccess : hipStreamSynchronize(stream);
        }
        std::vector<HostChunk> chunks;
        std::vector<char*> dev;
        for (const ArrayCopy& a : arrays)
        {
            if (a.bytes == 0) continue;
            // the runtime copies its own memory, whichever device's, without a slot
            if (reach(device, a.host, a.bytes, 1) != Reach::Host)
            {
                const hipError_t e = hipMemcpyAsync(up ? a.dev : a.host, up ? a.host : a.dev, a.bytes,
                                                    hipMemcpyDefault, stream);
                if (e != hipSuccess) return e;
                continue;
            }
            for (std::size_t o = 0; o < a.bytes; o += kSlot)
            {
                chunks.push_back(HostChunk{static_cast<char*>(a.host) + o, std::min(kSlot, a.bytes - o), Reach::Host});
                dev.push_back(static_cast<char*>(a.dev) + o);
            }
        }
        return run(device, stream, up, chunks, [&](int c, char* p) {
            return hipMemcpyAsync(up ? dev[c] : p, up ? p : dev[c], chunks[c].bytes, hipMemcpyDefault, stream);
        });
    }

    // The reach of a caller's array of elements of `size` bytes from a kernel on
    // `device`: the device's own memory, aligned and allocated over the whole array.
    static Reach reach(int device, const void* p, std::size_t bytes, std::size_t size)
    {
        hipPointerAttribute_t at{};
        const bool known = hipPointerGetAttributes(&at, p) == hipSuccess;
        Reach r = Reach::Host;
        if (known && (at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged || at.type == hipMemoryTypeUnified))
        {
            r = Reach::Runtime;
            hipDeviceptr_t base = nullptr;
            std::size_t n = 0;
            if (at.type == hipMemoryTypeDevice && at.device == device && reinterpret_cast<std::uintptr_t>(p) % size == 0 &&
                hipMemGetAddressRange(&base, &n, const_cast<void*>(p)) == hipSuccess)
            {
                const std::size_t o = std::size_t(static_cast<const char*>(p) - static_cast<const char*>(base));
                if (o <= n && bytes <= n - o) r = Reach::Kernel;
            }
        }
        hipGetLastError();  // an ordinary host array is no error
        return r;
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

    hipError_t prepare()
    {
        while (int(events_.size()) < kSlots)
        {
            hipEvent_t ev = nullptr;
            const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
            if (e != hipSuccess) return e;
            events_.push_back(ev);
        }
        if (slots_) return hipSuccess;
        const hipError_t e = hipHostMalloc(&slots_, kSlot * kSlots, 0);
        if (e != hipSuccess) slots_ = nullptr;
        return e;
    }

    std::mutex busy_;
    void* slots_ = nullptr;
    std::vector<hipEvent_t> events_;
};

}  // namespace nimbus
