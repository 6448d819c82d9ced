// The host transfers (transfer.hpp) on the CPU: the runtime's calls replaced by
// ones that succeed at once and the launches of the two layout kernels by loops
// over their chunks.  New threads can be held back before their first
// instruction (pthread_create below), as they are where another pool's threads
// spin on every processor.
//
//   transfer_threads held     every helper held until the transfers have returned
//   transfer_threads free N   helpers run at once; N rounds
// Both move q of several grids up and down and compare every value, ghost layers
// included; exit status 0 if all is right.
#include <hip/hip_runtime.h>

#include <dlfcn.h>
#include <pthread.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) emulate(#kernel, grid, __VA_ARGS__)
#define hipGetLastError() hipSuccess
#define hipSetDevice(d) hipSuccess
#define hipEventRecord(e, s) hipSuccess
#define hipEventSynchronize(e) hipSuccess
#define hipStreamSynchronize(s) hipSuccess

#include "kernels.hpp"

namespace howmhd {
// k_ref_to_dev, k_dev_to_ref: column (j, k) of nz values from y plane j0, x from i0
template <typename P, typename D>
void emulate(const char* kernel, dim3 grid, P a, D b, const Geom& g, int i0, int ni, int j0, int ncol) {
    const bool up = std::strcmp(kernel, "k_ref_to_dev") == 0;
    double* pin = const_cast<double*>(up ? a : b);
    double* dev = const_cast<double*>(up ? b : a);
    for (unsigned m = 0; m < grid.z; ++m)
        for (int x = 0; x < ni; ++x)
            for (int c = 0; c < ncol; ++c) {
                const size_t j = j0 + c / g.n[2], k = c % g.n[2];
                double& d = dev[(size_t)m * g.ncell + (k * g.n[1] + j) * g.n[0] + i0 + x];
                double& p = pin[((size_t)m * ni + x) * ncol + c];
                if (up) d = p;
                else p = d;
            }
}
}  // namespace howmhd

#include "transfer.hpp"

static std::atomic<bool> hold{false};
static std::atomic<int> created{0};

struct Start {
    void* (*fn)(void*);
    void* arg;
};
static void* held_start(void* p) {
    const Start s = *(Start*)p;
    delete (Start*)p;
    while (hold.load()) usleep(200);
    return s.fn(s.arg);
}
#if !__has_feature(thread_sanitizer)
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*fn)(void*), void* arg) {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
    ++created;
    return real(t, a, held_start, new Start{fn, arg});
}
#endif

using namespace howmhd;

static int image(int a, int n, int per) { return bmap(a, n, per); }

static bool round_trip(howmhd_gpu_ctx& c, int nvar) {
    const int* n = c.g.n;
    const size_t n6y = n[1] + 6, n6z = n[2] + 6, n6 = (n[0] + 6) * n6y * n6z;
    std::vector<double> ref(nvar * n6, -1.0), dev(nvar * c.ncell, -2.0), out(nvar * n6, -3.0);
    auto value = [&](int m, int i, int j, int k) { return m * 1e9 + i * 1e6 + j * 1e3 + k + 0.5; };
    auto at = [&](int m, int i, int j, int k) { return m * n6 + ((size_t)(i + 3) * n6y + j + 3) * n6z + k + 3; };
    for (int m = 0; m < nvar; ++m)
        for (int i = 0; i < n[0]; ++i)
            for (int j = 0; j < n[1]; ++j)
                for (int k = 0; k < n[2]; ++k) ref[at(m, i, j, k)] = value(m, i, j, k);
    if (transfer<true>(&c, ref.data(), dev.data(), nvar)) return false;
    if (transfer<false>(&c, out.data(), dev.data(), nvar)) return false;
    for (int m = 0; m < nvar; ++m)
        for (int i = -3; i < n[0] + 3; ++i)
            for (int j = -3; j < n[1] + 3; ++j)
                for (int k = -3; k < n[2] + 3; ++k) {
                    const int a = image(i, n[0], c.g.per[0]), b = image(j, n[1], c.g.per[1]), d = image(k, n[2], c.g.per[2]);
                    if (out[at(m, i, j, k)] != value(m, a, b, d)) {
                        std::printf("value %d %d %d %d\n", m, i, j, k);
                        return false;
                    }
                    if (i == a && j == b && k == d && dev[m * c.ncell + ((size_t)d * n[1] + b) * n[0] + a] != value(m, a, b, d))
                        return false;
                }
    return true;
}

int main(int argc, char** argv) {
    const bool held = argc > 1 && std::strcmp(argv[1], "held") == 0;
    const int grids[][3] = {{48, 40, 50}, {97, 75, 61}, {300, 280, 1}, {5, 3, 4000}, {20000, 1, 1}, {130, 100, 90}};
    const int rounds = argc > 2 ? std::atoi(argv[2]) : 1;
    for (int r = 0; r < rounds; ++r)
        for (const auto& n : grids) {
            howmhd_gpu_ctx c;
            for (int d = 0; d < 3; ++d) { c.g.n[d] = n[d]; c.g.per[d] = (r + d) % 2; }
            c.ncell = (size_t)n[0] * n[1] * n[2];
            c.g.ncell = (long long)c.ncell;
            c.xfer_slot = xfer_slot(c.ncell, n[2]);
            c.xfer_n = xfer_slots(c.ncell, c.xfer_slot);
            std::vector<double> slots(c.xfer_n * c.xfer_slot);
            c.xfer = slots.data();
            c.xfer_ev.assign(c.xfer_n, nullptr);
            hold = held;
            const bool ok = round_trip(c, 8) && round_trip(c, 3);
            hold = false;
            std::printf("%s %d x %d x %d: %s, %d threads so far\n", argv[1], n[0], n[1], n[2], ok ? "right" : "WRONG",
                        created.load());
            std::fflush(stdout);
            if (!ok) return 1;
        }
    return 0;
}
