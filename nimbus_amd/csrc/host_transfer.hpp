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
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace nimbus
{

// A contiguous piece of one of the caller's arrays; direct: the kernel can
// reach the array itself (device memory), nothing is copied.
struct HostChunk
{
    char* host;
    std::size_t bytes;
    bool direct;
};

class HostTransfer
{
public:
    static constexpr std::size_t kSlot = std::size_t(2) << 20;
    static constexpr int kSlots = 10;
    static constexpr int kThreads = 6;

    HostTransfer() = default;
    HostTransfer(const HostTransfer&) = delete;
    HostTransfer& operator=(const HostTransfer&) = delete;
    ~HostTransfer()
    {
        for (hipEvent_t e : events_) hipEventDestroy(e);
        if (slots_) hipHostFree(slots_);
    }

    // Moves the chunks to (up) or from the device; launch(c, p) enqueues the
    // device side of chunk c on `stream` against p, its slot or (direct) its
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
        std::size_t bytes = 0;
        for (const HostChunk& c : chunks) bytes += c.bytes;
        // a thread for each MB: below that starting one costs as much as it takes over
        const int want = int(std::min<std::size_t>({std::size_t(kThreads), chunks.size(), bytes >> 20}));
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
                    hipError_t r = launch(c, chunks[c].direct ? chunks[c].host : slot(c));
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
        if (r == hipSuccess && !k.direct)
        {
            if (up) std::memcpy(slot(c), k.host, k.bytes);
            else std::memcpy(k.host, slot(c), k.bytes);
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
