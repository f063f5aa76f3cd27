// csrc/host_counts.h on a host without a GPU: the HIP calls it makes are stood in for here, the "kernels" are threads.
// One check by name per run; exit status 0 if it holds.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "../umdk_original_amd/csrc/host_counts.h"

using cam_torch::HostCounts;

namespace {
std::atomic<int> g_allocated{0}, g_freed{0};
thread_local int t_device = 0;      // the current device, 0 as in a fresh thread
int g_device_at_malloc = -1;
unsigned g_flags = 0;
std::atomic<int> g_query{(int)hipErrorNotReady};

#define REQUIRE(c)                                              \
    do {                                                        \
        if (!(c)) {                                             \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                       \
        }                                                       \
    } while (0)

bool throws(HostCounts &c, int64_t *out)
{
    try {
        c.wait(nullptr, out);
    } catch (const std::runtime_error &) {
        return true;
    }
    return false;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d)
{
    *d = t_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    t_device = d;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    g_device_at_malloc = t_device;
    g_flags = flags;
    ++g_allocated;
    *p = std::malloc(bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    ++g_freed;
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return (hipError_t)g_query.load(); }
const char *hipGetErrorString(hipError_t) { return "an error"; }
}

static void device()
{
    // the tensors' device, not the current one; usable from the others later; the current one is what it was
    HostCounts c(3, 5);
    REQUIRE(g_device_at_malloc == 5 && t_device == 0);
    REQUIRE((g_flags & hipHostMallocPortable) && (g_flags & hipHostMallocCoherent));
    HostCounts other(512, 2);
    REQUIRE(g_allocated == 1 && t_device == 0);
}

static void arrive()
{
    HostCounts c(512, 0);
    int64_t *p = c.data();
    for (int i = 0; i < 512; ++i) {
        REQUIRE(p[i] == -1);
    }
    c.queued();
    std::thread kernel([p] {
        for (int i = 511; i >= 0; --i) {
            std::this_thread::sleep_for(std::chrono::microseconds(20));
            ((volatile int64_t *)p)[i] = i % 7;
        }
    });
    int64_t out[512];
    c.wait(nullptr, out);
    kernel.join();
    for (int i = 0; i < 512; ++i) {
        REQUIRE(out[i] == i % 7);
    }
}

static void threads()
{
    int64_t *mine, *theirs = nullptr;
    HostCounts c(4, 0);
    mine = c.data();
    std::thread([&theirs] {
        HostCounts d(4, 1);
        theirs = d.data();
        REQUIRE(t_device == 0);
    }).join();
    REQUIRE(theirs != nullptr && theirs != mine && g_allocated == 2 && g_freed == 1);  // given back with its thread
}

static void errors()
{
    int64_t out[4];
    {
        HostCounts c(4, 0);
        c.data()[0] = 1;
        g_query = (int)hipErrorNotReady;
        c.queued();
        g_query = (int)hipSuccess;    // the stream is done, three counts never came
        REQUIRE(throws(c, out));
    }
    {
        HostCounts c(4, 0);
        g_query = (int)hipErrorUnknown;
        c.queued();
        REQUIRE(throws(c, out));
    }
    {
        HostCounts c(0, 0);   // nothing to wait for
        REQUIRE(!throws(c, out));
    }
    bool refused = false;
    try {
        HostCounts c(513, 0);
    } catch (const std::runtime_error &) {
        refused = true;
    }
    REQUIRE(refused);
}

static void late()
{
    // a call that fails behind its launch: its kernel still stores, and the next call must not take that for its own
    int64_t *old;
    {
        HostCounts c(2, 0);
        old = c.data();
        c.queued();
    }
    HostCounts c(2, 0);
    REQUIRE(c.data() != old);
    old[0] = old[1] = 9;
    REQUIRE(c.data()[0] == -1 && c.data()[1] == -1);
    // one that fails before: the buffer stays
    int64_t *kept = c.data();
    {
        HostCounts d(2, 0);
    }
    REQUIRE(HostCounts(2, 0).data() == kept && g_allocated == 2);
}

int main(int argc, char **argv)
{
    REQUIRE(argc == 2);
    const struct {
        const char *name;
        void (*fn)();
    } checks[] = {{"device", device}, {"arrive", arrive}, {"threads", threads}, {"errors", errors}, {"late", late}};
    for (const auto &c : checks) {
        if (std::strcmp(c.name, argv[1]) == 0) {
            c.fn();
            return 0;
        }
    }
    return 2;
}
