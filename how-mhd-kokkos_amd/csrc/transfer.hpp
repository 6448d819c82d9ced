// Host transfers: the caller's arrays in the reference layout (m, i, j, k)
// with three ghost layers per side <-> the device layout (m, z, y, x) of
// active cells.
//
// Only active cells cross PCIe.  A transfer is cut into chunks that fit a
// pinned slot of the context: whole variables, or a range of y planes of one,
// or a range of x of one y plane.  A chunk lies in its slot as (m, i, j, k)
// without ghosts.  Host threads move chunks between the caller's (pageable)
// memory and their slots, filling the ghost layers with their images on the
// way down, while the transpose kernel reads or writes the other slots of the
// pinned memory over PCIe; on large grids there are two slots a thread, so that
// its copy overlaps its kernel.  A thread that comes late finds less to do, or
// nothing (helpers.hpp).
//
// Bound: PCIe (56 GB/s each way) for large grids, the first touch of the
// caller's pages on the way down, the start of the threads and one chunk's
// latency for small ones.  q(0) up and down, against one variable at a time
// through the runtime's pageable copies, ghosts included: 256^3 (1.15 GB)
// 39 -> 23 and 111 -> 35 ms, 512x512 4.2 -> 0.96 and 11.9 -> 3.3 ms, 48x40x50
// 0.42 -> 0.37 and 0.74 -> 0.38 ms, 32^3 0.24 -> 0.16 and 0.37 -> 0.19 ms.
#pragma once

#include "context.hpp"
#include "tstep_kernels.hpp"

#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace howmhd {
namespace {

constexpr int kXferThreads = 8, kXferChunks = 2 * kXferThreads, kXferSlots = 2 * kXferThreads;
constexpr size_t kXferSlotMax = 1u << 18, kXferSlotMin = 1u << 15;  // values: 2 MiB, 256 KiB

// Values per slot of a context of ncell cells: eight variables in 16 chunks,
// within the bounds; a row of nz values fits.  (32 chunks: 48x40x50 up in 0.52
// instead of 0.36 ms, because the chunks' kernels follow one another.)
inline size_t xfer_slot(size_t ncell, int nz) {
    return std::max(std::min(std::max(8 * ncell / kXferChunks, kXferSlotMin), kXferSlotMax), (size_t)nz);
}
// Slots: two a thread where the chunks are at their bound and every thread
// moves many (144^3 down in 5.7 instead of 6.9 ms); else one, which costs the
// transfer nothing and halves the memory that create pins and the first
// transfer touches (64^3: first upload 1.20 against 1.58 ms).
inline int xfer_slots(size_t ncell, size_t slot) {
    const size_t most = slot < kXferSlotMax ? kXferThreads : kXferSlots;
    return (int)std::min(most, (8 * ncell + slot - 1) / slot);
}

struct Chunk {
    int m0, nm, i0, ni, j0, nj;
};

// The chunks of nvar variables.
inline std::vector<Chunk> xfer_chunks(const Geom& g, int nvar, size_t slot) {
    const size_t nx = g.n[0], ny = g.n[1], nz = g.n[2], nc = nx * ny * nz;
    // n in the fewest equal parts of at most `most`
    auto even = [](size_t n, size_t most) {
        const size_t parts = (n + std::max<size_t>(1, most) - 1) / std::max<size_t>(1, most);
        return (int)((n + parts - 1) / parts);
    };
    const int dm = even(nvar, slot / nc);
    const int dj = even(ny, slot / (nx * nz));
    const int di = even(nx, slot / nz);
    std::vector<Chunk> v;
    for (int m = 0; m < nvar; m += dm)
        for (int j = 0; j < (int)ny; j += dj)
            for (int i = 0; i < (int)nx; i += di)
                v.push_back({m, std::min(dm, nvar - m), i, std::min(di, (int)nx - i), j, std::min(dj, (int)ny - j)});
    return v;
}

// Padded indices (0..n+5) whose value is that of active index a: its own, and
// the ghosts that map to it (at most 6).
inline int images(int a, int n, int per, int* out) {
    int k = 0;
    out[k++] = a + 3;
    if (a < 3 || a >= n - 3)
        for (int q = 0; q < 6; ++q) {
            const int p = q < 3 ? q : n + q;
            if (bmap(p - 3, n, per) == a) out[k++] = p;
        }
    return k;
}

// The chunk's active cells from the caller's array into a slot.
inline void pack(const Geom& g, const double* ref, const Chunk& c, double* slot) {
    const size_t n6y = (size_t)g.n[1] + 6, n6z = (size_t)g.n[2] + 6, n6 = ((size_t)g.n[0] + 6) * n6y * n6z;
    const size_t nz = g.n[2];
    for (int m = c.m0; m < c.m0 + c.nm; ++m)
        for (int i = c.i0; i < c.i0 + c.ni; ++i) {
            const double* s = ref + m * n6 + (((size_t)i + 3) * n6y + c.j0 + 3) * n6z + 3;
            if (nz == 1) {
                for (int j = 0; j < c.nj; ++j) slot[j] = s[j * n6z];
                slot += c.nj;
            } else {
                for (int j = 0; j < c.nj; ++j, s += n6z, slot += nz) std::memcpy(slot, s, nz * sizeof(double));
            }
        }
}

// A slot's cells into the caller's array, with every ghost cell whose image
// is one of them.
inline void unpack(const Geom& g, const double* slot, const Chunk& c, double* ref) {
    const size_t n6y = (size_t)g.n[1] + 6, n6z = (size_t)g.n[2] + 6, n6 = ((size_t)g.n[0] + 6) * n6y * n6z;
    const int nz = g.n[2];
    int lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = bmap(k - 3, nz, g.per[2]);
        hi[k] = bmap(nz + k, nz, g.per[2]);
    }
    int im[7], jm[7];
    for (int m = c.m0; m < c.m0 + c.nm; ++m)
        for (int i = c.i0; i < c.i0 + c.ni; ++i) {
            const int ki = images(i, g.n[0], g.per[0], im);
            for (int j = c.j0; j < c.j0 + c.nj; ++j, slot += nz) {
                const int kj = images(j, g.n[1], g.per[1], jm);
                for (int a = 0; a < ki; ++a)
                    for (int b = 0; b < kj; ++b) {
                        double* d = ref + m * n6 + ((size_t)im[a] * n6y + jm[b]) * n6z;
                        for (int k = 0; k < 3; ++k) d[k] = slot[lo[k]];
                        std::memcpy(d + 3, slot, nz * sizeof(double));
                        for (int k = 0; k < 3; ++k) d[nz + 3 + k] = slot[hi[k]];
                    }
            }
        }
}

// Processors this process may run on.
inline int cpu_share() {
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof(set), &set) == 0) return std::max(1, CPU_COUNT(&set));
    return std::max(1u, std::thread::hardware_concurrency());
}

// Moves nvar variables between ref (host) and dev; synchronises.
template <bool UP>
int transfer(howmhd_gpu_ctx* c, double* ref, double* dev, int nvar) {
    const Geom& g = c->g;
    const size_t n6 = ((size_t)g.n[0] + 6) * ((size_t)g.n[1] + 6) * ((size_t)g.n[2] + 6);
    std::vector<Chunk> chunks;
    try {
        chunks = xfer_chunks(g, nvar, c->xfer_slot);
    } catch (const std::bad_alloc&) {
        return fail(c, HOWMHD_ENOMEM, "host transfer: out of host memory");
    }
    // threads where they have a MiB of the caller's memory each, two chunks in flight for each
    const size_t bytes = nvar * n6 * sizeof(double);
    const int nw = (int)std::max<size_t>(1, std::min<size_t>({(size_t)cpu_share(), kXferThreads, chunks.size(), bytes >> 20,
                                                              (size_t)c->xfer_n}));
    const int most = 2 * nw;
    // Under the mutex: the next chunk, the free slots (a bit each), the slots
    // with a chunk in flight, oldest first, and the first error.  A thread is
    // at one slot at a time; any thread may finish any chunk in flight.
    std::mutex mu;
    size_t next = 0;
    unsigned idle = (1u << c->xfer_n) - 1;
    struct {
        int slot;
        size_t chunk;
    } flight[kXferSlots];
    int first = 0, flying = 0;
    hipError_t err = hipSuccess;
    const char* what = "";
    auto report = [&](hipError_t e, const char* w) {
        std::lock_guard<std::mutex> lk(mu);
        if (err == hipSuccess) { err = e; what = w; }
        (void)hipGetLastError();
    };
    auto launch = [&](const Chunk& k, int slot) {
        const int ncol = k.nj * g.n[2];
        const dim3 grid(blocks_for(ncol, LAY_T), blocks_for(k.ni, LAY_T), k.nm);
        double* pin = c->xfer + (size_t)slot * c->xfer_slot;
        double* d = dev + (size_t)k.m0 * c->ncell;
        if (UP) hipLaunchKernelGGL(k_ref_to_dev, grid, dim3(256), 0, c->stream, (const double*)pin, d, g, k.i0, k.ni, k.j0, ncol);
        else hipLaunchKernelGGL(k_dev_to_ref, grid, dim3(256), 0, c->stream, (const double*)d, pin, g, k.i0, k.ni, k.j0, ncol);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(c->xfer_ev[slot], c->stream);
        if (e != hipSuccess) report(e, "launch");
        return e == hipSuccess;
    };
    auto arrived = [&](int slot) {
        const hipError_t e = hipEventSynchronize(c->xfer_ev[slot]);
        if (e != hipSuccess) report(e, "hipEventSynchronize");
        return e == hipSuccess;
    };
    auto work = [&](bool helper) {
        if (helper && hipSetDevice(c->device) != hipSuccess) return report(hipErrorInvalidDevice, "hipSetDevice");
        for (;;) {
            int slot;
            size_t k;
            bool fill;
            {
                std::lock_guard<std::mutex> lk(mu);
                const bool more = next < chunks.size();
                fill = more && idle != 0 && flying < most;
                if (err != hipSuccess) return;
                if (fill) {
                    slot = __builtin_ctz(idle);
                    idle &= idle - 1;
                    k = next++;
                } else if (flying > 0 && (more || !UP)) {  // (up, the stream's end ends the last ones)
                    slot = flight[first].slot;
                    k = flight[first].chunk;
                    first = (first + 1) % kXferSlots;
                    --flying;
                } else {
                    return;  // no more threads than slots: what is left is in other threads' hands
                }
            }
            if (fill) {
                if (UP) pack(g, ref, chunks[k], c->xfer + (size_t)slot * c->xfer_slot);
                if (!launch(chunks[k], slot)) return;
                std::lock_guard<std::mutex> lk(mu);
                flight[(first + flying++) % kXferSlots] = {slot, k};
            } else {
                if (!arrived(slot)) return;
                if (!UP) unpack(g, c->xfer + (size_t)slot * c->xfer_slot, chunks[k], ref);
                std::lock_guard<std::mutex> lk(mu);
                idle |= 1u << slot;
            }
        }
    };
    c->xfer_helpers.run(nw - 1, work);
    if (err != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);
        return fail(c, HOWMHD_EHIP, std::string("host transfer: ") + what + ": " + hipGetErrorString(err));
    }
    HCHECK(c, hipStreamSynchronize(c->stream));
    return HOWMHD_OK;
}

// A caller's pointer to device memory is not the documented use, but a copy
// accepts it: it goes through host memory.
inline bool on_device(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // ordinary host memory
        return false;
    }
    return a.type == hipMemoryTypeDevice;
}

inline int upload_ref(howmhd_gpu_ctx* c, const double* ref, double* dev, int nvar) {
    if (!on_device(ref)) return transfer<true>(c, const_cast<double*>(ref), dev, nvar);
    try {
        std::vector<double> host((size_t)nvar * (c->g.n[0] + 6) * (c->g.n[1] + 6) * (c->g.n[2] + 6));
        HCHECK(c, hipMemcpy(host.data(), ref, host.size() * sizeof(double), hipMemcpyDeviceToHost));
        return transfer<true>(c, host.data(), dev, nvar);
    } catch (const std::bad_alloc&) {
        return fail(c, HOWMHD_ENOMEM, "host transfer: out of host memory");
    }
}

inline int download_ref(howmhd_gpu_ctx* c, double* dev, double* ref, int nvar) {
    if (!on_device(ref)) return transfer<false>(c, ref, dev, nvar);
    try {
        std::vector<double> host((size_t)nvar * (c->g.n[0] + 6) * (c->g.n[1] + 6) * (c->g.n[2] + 6));
        const int rc = transfer<false>(c, host.data(), dev, nvar);
        if (rc) return rc;
        HCHECK(c, hipMemcpy(ref, host.data(), host.size() * sizeof(double), hipMemcpyHostToDevice));
        return HOWMHD_OK;
    } catch (const std::bad_alloc&) {
        return fail(c, HOWMHD_ENOMEM, "host transfer: out of host memory");
    }
}

}  // namespace
}  // namespace howmhd
