// The host transfers of slgpu_hostio.h on a HIP runtime of a few lines: "device" memory is host
// memory, copies happen at the call, events are complete at once.  Prints one line per check and exits
// with the number of failures.
#include "../../superlite_amd/csrc/slgpu_hostio.h"

#include <cstdio>
#include <dirent.h>
#include <sched.h>

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) { *p = malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned int) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t);
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}

static int failures = 0, most_threads = 0;

static int threads()
{
    int n = 0;
    DIR *d = opendir("/proc/self/task");
    while (dirent *e = readdir(d)) n += e->d_name[0] != '.';
    closedir(d);
    return n;
}

hipError_t hipEventSynchronize(hipEvent_t)
{
    most_threads = std::max(most_threads, threads());
    return hipSuccess;
}

static void check(bool ok, const char *what, size_t n)
{
    printf("%s %s %zu\n", ok ? "ok" : "FAILED", what, n);
    fflush(stdout);
    failures += !ok;
}

int main()
{
    using namespace slgpu;
    cpu_set_t all;
    if (sched_getaffinity(0, sizeof(all), &all) != 0) return 98;
    for (int cores : {CPU_COUNT(&all), std::min(2, CPU_COUNT(&all)), 1})
    for (size_t n : {(size_t)1, (size_t)4096, (size_t)1048575, (size_t)1048576, (size_t)2097153, (size_t)30000001}) {
        cpu_set_t s;
        CPU_ZERO(&s);
        for (int k = 0; k < CPU_SETSIZE && CPU_COUNT(&s) < cores; ++k)
            if (CPU_ISSET(k, &all)) CPU_SET(k, &s);
        sched_setaffinity(0, sizeof(s), &s);
        most_threads = 0;
        HostIO io;
        if (io.create(4096, n) != hipSuccess) return 99;
        std::vector<char> dev(n + 77), a(n, 0), b(77, 0);
        for (size_t k = 0; k < dev.size(); ++k) dev[k] = (char)(k * 2654435761u >> 13);
        const auto t0 = std::chrono::steady_clock::now();
        {
            Outputs out(io, nullptr);
            out.add(a.data(), dev.data(), n);
            out.add(b.data(), dev.data() + n, 77, true);
            out.start();
            check(out.finish(nullptr) == hipSuccess, "finish", n);
            const double wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
            check(memcmp(a.data(), dev.data(), n) == 0 && memcmp(b.data(), dev.data() + n, 77) == 0, "bytes", n);
            // events here are complete before the copies out of the ring begin
            check(out.tail_ms() > 0.0 && out.tail_ms() <= wall, "tail", n);
        }
        // at most eight threads beside the caller's, each with a MiB to copy and a core to run on
        const size_t most = std::min<size_t>({8, (n + 77) >> 20, (size_t)CPU_COUNT(&s) - 1});
        check(most_threads <= 1 + (int)most, "threads", n);
        io.destroy();
    }
    return failures;
}
