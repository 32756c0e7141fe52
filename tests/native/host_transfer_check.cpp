// Checks of nimbus_amd/csrc/host_transfer.hpp without a GPU, against the
// runtime interface in hip_on_host. One check per run, named by the argument.
#include "host_transfer.hpp"

#include <cstdio>
#include <new>
#include <string>

// Allocations fail from the `fail_in`-th of the thread that sets it on.
namespace
{
thread_local int fail_in = 0;
}

void* operator new(std::size_t n)
{
    if (fail_in > 0 && --fail_in == 0)
    {
        fail_in = 1;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

using namespace nimbus;

#define CHECK(x)                                                        \
    do                                                                  \
    {                                                                   \
        if (!(x))                                                       \
        {                                                               \
            std::printf("line %d: %s\n", __LINE__, #x);                 \
            return 1;                                                   \
        }                                                               \
    } while (0)

namespace
{
constexpr std::size_t KB = 1024, MB = 1024 * KB;

// n arrays of `bytes` and their device copies, both of distinct contents.
struct Arrays
{
    std::vector<std::vector<char>> host, dev;
    std::vector<ArrayCopy> copies;
    Arrays(int n, std::size_t bytes)
    {
        for (int q = 0; q < n; ++q)
        {
            host.emplace_back(bytes);
            dev.emplace_back(bytes);
            for (std::size_t b = 0; b < bytes; ++b)
            {
                host[q][b] = char(b * 7 + q);
                dev[q][b] = char(b * 11 + q + 3);
            }
        }
        for (int q = 0; q < n; ++q) copies.push_back(ArrayCopy{dev[q].data(), host[q].data(), bytes});
    }
    bool equal() const { return host == dev; }
};

// Small calls take one plain copy per array: no ring, no events, no queries.
int small()
{
    for (bool up : {true, false})
        for (std::size_t bytes : {std::size_t(0), std::size_t(1), 100 * KB, 512 * KB - 1})
        {
            HostTransfer t;
            Arrays a(up ? 13 : 16, bytes);
            fake::reset();
            CHECK(t.copy(0, nullptr, up, a.copies) == hipSuccess);
            CHECK(a.equal());
            CHECK(fake::copies == (bytes ? int(a.copies.size()) : 0));
            CHECK(fake::pinned == 0 && fake::events == 0 && fake::threads_set == 0 && fake::queries == 0);
        }
    return 0;
}

// Large ones take the ring, also with lengths that are no multiple of a slot.
int large()
{
    for (bool up : {true, false})
    {
        HostTransfer t;
        Arrays a(8, 7 * MB + 13);
        fake::reset();
        CHECK(t.copy(0, nullptr, up, a.copies) == hipSuccess);
        CHECK(a.equal());
        CHECK(fake::pinned == 1 && fake::events == 8 * 4);
        CHECK(fake::pinned_flags & hipHostMallocCoherent);
    }
    return 0;
}
// A kernel on the context's device (0) touches only memory of that device and
// host memory pinned for it, over its whole allocation, aligned; what else the
// runtime knows it copies itself, but for pinned memory, which the host can.
int reach()
{
    std::vector<char> a(64 * KB);
    char* const p = a.data();
    auto how = [&](std::size_t shift, std::size_t bytes, std::size_t size) {
        return HostTransfer::place(0, p + shift, bytes, size).reach;
    };
    CHECK(how(0, 4 * KB, 4) == Reach::Host && !HostTransfer::of_runtime(p));
    for (hipMemoryType type : {hipMemoryTypeDevice, hipMemoryTypeHost, hipMemoryTypeManaged})
        for (int device : {0, 1})
        {
            fake::ranges = {{p, fake::Range{64 * KB, type, device}}};
            const Reach other = type == hipMemoryTypeHost ? Reach::Host : Reach::Runtime;
            const Reach own = device == 0 && type != hipMemoryTypeManaged ? Reach::Kernel : other;
            CHECK(HostTransfer::of_runtime(p));
            CHECK(how(0, 64 * KB, 4) == own);
            CHECK(how(4 * KB, 60 * KB, 8) == own);
            CHECK(how(4 * KB, 60 * KB + 1, 4) == other);
            CHECK(how(2, 4 * KB, 4) == other);
            CHECK(how(4, 4 * KB, 8) == other);
        }
    // pinned memory has an address of its own on the device
    fake::ranges = {{p, fake::Range{64 * KB, hipMemoryTypeHost, 0}}};
    fake::mapped = 1 << 20;
    const bool at = HostTransfer::place(0, p + 8, 4 * KB, 8).at == p + 8 + fake::mapped;
    const bool on_host = HostTransfer::place(0, p + 4, 4 * KB, 8).at == p + 4;
    fake::mapped = 0;
    CHECK(at && on_host);
    return 0;
}

// Whole arrays in pinned memory take plain copies at any size: no ring, no threads.
int pinned()
{
    for (bool up : {true, false})
    {
        HostTransfer t;
        Arrays a(8, 7 * MB + 13);
        fake::ranges.clear();
        for (auto& h : a.host) fake::ranges[h.data()] = fake::Range{h.size(), hipMemoryTypeHost, 0};
        fake::reset();
        CHECK(t.copy(0, nullptr, up, a.copies) == hipSuccess);
        CHECK(a.equal());
        CHECK(fake::copies == 8 && fake::pinned == 0 && fake::events == 0 && fake::threads_set == 0);
    }
    return 0;
}

// Another device's array goes through the slots with the runtime's copies, and
// in a copy of whole arrays without them.
int foreign()
{
    for (bool up : {true, false})
    {
        Arrays a(8, 7 * MB + 13);
        fake::ranges = {{a.host[3].data(), fake::Range{a.host[3].size(), hipMemoryTypeDevice, 1}}};
        {
            HostTransfer t;
            fake::reset();
            CHECK(t.copy(0, nullptr, up, a.copies) == hipSuccess);
            CHECK(a.equal());
            CHECK(fake::events == 7 * 4 && fake::copies == 7 * 4 + 1 && fake::blocking_copies == 0);
        }
        HostTransfer t;
        std::vector<char> from(3 * MB, 5), to(3 * MB, 6);
        const std::vector<HostChunk> chunks{{(up ? from : to).data(), MB, Reach::Host},
                                            {(up ? from : to).data() + MB, 2 * MB, Reach::Runtime}};
        char* const dev = (up ? to : from).data();
        fake::reset();
        CHECK(t.run(0, nullptr, up, chunks, [&](int c, char* p) {
            char* const d = dev + (c ? MB : 0);
            return hipMemcpyAsync(up ? d : p, up ? p : d, chunks[c].bytes, hipMemcpyDefault, nullptr);
        }) == hipSuccess);
        CHECK(to == from && fake::blocking_copies == 1);
    }
    return 0;
}
// Arrays that share memory hold what the last of them is given, as plain copies
// in order leave it.
int shared()
{
    for (std::size_t shift : {std::size_t(0), MB})
        for (int repeat = 0; repeat < 20; ++repeat)
        {
            HostTransfer t;
            Arrays a(16, 2 * MB);
            std::vector<char> sink(2 * MB + 15 * shift, 1), expect(sink);
            for (int q = 0; q < 16; ++q)
            {
                a.copies[q].host = sink.data() + q * shift;
                std::memcpy(expect.data() + q * shift, a.dev[q].data(), 2 * MB);
            }
            CHECK(t.copy(0, nullptr, false, a.copies) == hipSuccess);
            CHECK(sink == expect);
        }
    return 0;
}

// Memory that runs out while the team starts: the threads that did start, and
// the caller, move the arrays.
int no_memory()
{
    for (bool up : {true, false})
        for (int n = 1; n < 12; ++n)
        {
            HostTransfer t;
            std::vector<char> array(32 * MB, 1), dev(32 * MB, 2);
            std::vector<HostChunk> chunks;
            for (int c = 0; c < 16; ++c) chunks.push_back(HostChunk{array.data() + c * 2 * MB, 2 * MB, Reach::Host});
            auto launch = [&](int c, char* p) {
                char* const d = dev.data() + c * 2 * MB;
                return hipMemcpyAsync(up ? d : p, up ? p : d, chunks[c].bytes, hipMemcpyDefault, nullptr);
            };
            CHECK(t.run(0, nullptr, up, chunks, launch) == hipSuccess);  // makes the ring
            for (auto& b : up ? dev : array) b = 3;
            fake::reset();
            bool moved = true;
            fail_in = n;
            try
            {
                moved = t.run(0, nullptr, up, chunks, launch) == hipSuccess;
            }
            catch (const std::bad_alloc&)
            {
                moved = false;  // before any thread ran
            }
            fail_in = 0;
            CHECK(moved ? array == dev : fake::threads_set == 0 && fake::copies == 0);
        }
    return 0;
}

// Arrays that the kernel reaches itself need no copying thread.
int no_threads()
{
    for (bool up : {true, false})
    {
        HostTransfer t;
        std::vector<char> array(64 * MB, 1), dev(64 * MB, 2);
        std::vector<HostChunk> chunks;
        for (int c = 0; c < 4; ++c) chunks.push_back(HostChunk{array.data() + c * 16 * MB, 16 * MB, Reach::Kernel});
        fake::reset();
        CHECK(t.run(0, nullptr, up, chunks, [&](int c, char* p) {
            char* const d = dev.data() + c * 16 * MB;
            return hipMemcpyAsync(up ? d : p, up ? p : d, chunks[c].bytes, hipMemcpyDefault, nullptr);
        }) == hipSuccess);
        CHECK(array == dev && fake::copies == 4 && fake::threads_set == 0 && fake::pinned == 0);
    }
    return 0;
}
}  // namespace

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "small") return small();
    if (what == "large") return large();
    if (what == "no_threads") return no_threads();
    if (what == "no_memory") return no_memory();
    if (what == "shared") return shared();
    if (what == "pinned") return pinned();
    if (what == "reach") return reach();
    if (what == "foreign") return foreign();
    std::printf("unknown check %s\n", what.c_str());
    return 2;
}
