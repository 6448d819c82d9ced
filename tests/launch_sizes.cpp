// The launches of a stage, without a GPU: the launch code itself (stage.hpp)
// with the launch macro replaced by one that records name, grid and arguments.
// For each grid "nx,ny,nz,open,form" on the command line (open: 0 periodic; form:
// fp64, fp32, with i: routed; built with HOWMHD_EXACT=1 for fp64, 0 for fp32) it
// prints one line per launch,
//   name gridx gridy gridz blockx first_block
// then "tiles" with the tiles of each sweep axis as the kernel decodes them from
// the sweeps' blocks: "tiles axis expected covered twice" ("-" in place of the
// counts for a grid above 2^27 blocks, whose launches are only listed).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) record(#kernel, grid, block, __VA_ARGS__)
#define hipGetLastError() hipSuccess

namespace howmhd {
template <typename... A>
void record(const char* name, dim3 grid, dim3 block, const A&... args);
}

#include "kernels.hpp"
#include "stage.hpp"

namespace howmhd {

struct Axis {
    unsigned gx, gy, chunk, blocks;
    int first, march;
};
struct Launch {
    std::string name;
    dim3 grid, block;
    unsigned long long first;   // of the launch, from the sweeps' first block
    std::vector<Axis> axes;     // y, z, x of the sweeps
};
static std::vector<Launch> launches;
// (the reference-rounding form's IEEE-division launch takes its tiles from a queue)
static bool is_sweep(const Launch& l) {
    return l.name.find("k_sweep") != std::string::npos && !(HOWMHD_EXACT && l.name.find("DIV_IEEE") != std::string::npos);
}

template <typename A>
unsigned long long first_block(const A&, ...) { return 0; }
template <typename A>
auto first_block(const A& a, int) -> decltype((void)a.ax, 0ull) { return (unsigned long long)-(long long)a.ax[0].first; }

template <typename A>
void note_axes(const A&, ...) {}
template <typename A>
auto note_axes(const A& a, int) -> decltype((void)a.ax) {
    for (const auto& x : a.ax)
        launches.back().axes.push_back({x.gx, x.gy, x.by_chunk.d, x.by_blocks.d, (int)x.first, x.march});
}

template <typename... A>
void record(const char* name, dim3 grid, dim3 block, const A&... args) {
    launches.push_back({name, grid, block, 0, {}});
    ((launches.back().first = first_block(args, 0)), ...);
    (note_axes(args, 0), ...);
}

// The tiles of the axes, each decoded from the launches' blocks as the kernels do.
static void cover(bool split, const int* n) {
    const int dir[3] = {1, 2, 0};
    std::vector<unsigned char> seen[3];
    for (const Launch& l : launches) {
        if (!is_sweep(l)) continue;
        const std::vector<Axis>& axes = l.axes;
        for (int k = 0; k < 3; ++k)
            if (n[dir[k]] > 1) seen[k].resize((size_t)axes[k].gx * axes[k].gy);
        for (unsigned i = 0; i < l.grid.x; ++i) {
            const int b = (int)i;
            const int k = b >= axes[2].first ? 2 : b >= axes[1].first ? 1 : 0;
            const Axis& x = axes[k];
            const unsigned L = (unsigned)(b - x.first);
            auto mark = [&](unsigned bx, unsigned by) {
                if (bx < x.gx && by < x.gy) seen[k][bx + (size_t)x.gx * by]++;
            };
            if (split || k == 2) mark(L % x.gx, L / x.gx);  // (x tiles: a permutation of these)
            else {
                const unsigned r = L / x.chunk, hi = r / x.blocks;
                const unsigned bx = hi * x.chunk + (L - r * x.chunk), by = (r - hi * x.blocks) * x.march;
                for (int s = 0; s < x.march; ++s) mark(bx, by + s);
            }
        }
    }
    for (int k = 0; k < 3; ++k) {
        size_t once = 0, more = 0;
        for (unsigned char v : seen[k]) { once += v == 1; more += v > 1; }
        std::printf("tiles %c %zu %zu %zu\n", "xyz"[dir[k]], seen[k].size(), once, more);
    }
}

}  // namespace howmhd

int main(int argc, char** argv) {
    using namespace howmhd;
    for (int i = 1; i < argc; ++i) {
        howmhd_gpu_ctx c;
        int open = 0;
        char form[16] = "";
        if (std::sscanf(argv[i], "%d,%d,%d,%d,%15s", &c.g.n[0], &c.g.n[1], &c.g.n[2], &open, form) != 5) return 2;
        const int* n = c.g.n;
        for (int d = 0; d < 3; ++d) c.g.per[d] = !open;
        c.ncell = (size_t)n[0] * n[1] * n[2];
        c.g.ncell = (long long)c.ncell;
        c.p.dx = c.p.dy = c.p.dz = 1.0;
        c.ctf.use_x = n[0] > 1; c.ctf.use_y = n[1] > 1; c.ctf.use_z = n[2] > 1;
        c.ctf.use_Ox = c.ctf.use_x && c.ctf.use_y;
        c.ctf.use_Oy = c.ctf.use_y && c.ctf.use_z;
        c.ctf.use_Oz = c.ctf.use_x && c.ctf.use_z;
        c.ctf.active = c.ctf.use_Ox || c.ctf.use_Oy || c.ctf.use_Oz;
        c.plane = n[0] > 1 && n[1] > 1 && n[2] == 1;
        c.xlanes = x_lanes(c.g);
        c.route_now = std::strchr(form, 'i') != nullptr;
        launches.clear();
        std::printf("grid %s\n", argv[i]);
        const int rc = std::strncmp(form, "fp32", 4) == 0 ? launch_stage<float>(&c, 1, 1e-3) : launch_stage<double>(&c, 1, 1e-3);
        if (rc) { std::printf("error %s\n", c.err.c_str()); return 1; }
        unsigned long long nb = 0;
        bool split = false;
        for (const Launch& l : launches) {
            std::string name = l.name;
            name.erase(std::remove_if(name.begin(), name.end(), [](char ch) { return ch == ' ' || ch == '(' || ch == ')'; }),
                       name.end());
            std::printf("launch %s %u %u %u %u %llu\n", name.c_str(), l.grid.x, l.grid.y, l.grid.z,
                        l.block.x, l.first);
            if (is_sweep(l)) nb += l.grid.x;
            split = split || l.name.find("k_sweep_split") != std::string::npos;
        }
        if (nb <= 1u << 27) cover(split, n);
        else std::printf("tiles -\n");
    }
    return 0;
}
