// Checks of nimbus_amd/csrc/host_transfer.hpp without a GPU, against the
// runtime interface in hip_on_host. One check per run, named by the argument.
#include "host_transfer.hpp"

#include <cstdio>
#include <string>

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
    }
    return 0;
}
}  // namespace

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "small") return small();
    if (what == "large") return large();
    std::printf("unknown check %s\n", what.c_str());
    return 2;
}
