// Launch sequence of one SSPRK(5,4) stage (src/ssprk.cpp:1277-1329 with
// fluxct, src/fluxct.cpp:753-899).  Included by each translation unit of the
// library; the kernels it launches carry EX = HOWMHD_EXACT of that unit.
#pragma once

#include "context.hpp"

#include <algorithm>

namespace howmhd {
// internal linkage: each translation unit keeps its own copy (the units
// differ in HOWMHD_EXACT and contraction)
namespace {

constexpr int EX = HOWMHD_EXACT;

struct RK {
    double k1, k2, k3, k4, k5;
};

// SSPRK(5,4) coefficients, src/ssprk.cpp:66-94
inline RK rk_coeff(int iw) {
    RK c{0.0, 0.0, 0.0, 0.0, 0.0};
    switch (iw) {
    case 1: c.k1 = 1.0; c.k2 = 0.39175222700392; c.k3 = 0.0; break;
    case 2: c.k1 = 0.44437049406734; c.k2 = 0.36841059262959; c.k3 = 0.55562950593266; break;
    case 3: c.k1 = 0.62010185138540; c.k2 = 0.25189177424738; c.k3 = 0.37989814861460; break;
    case 4: c.k1 = 0.17807995410773; c.k2 = 0.54497475021237; c.k3 = 0.82192004589227; break;
    case 5:
        c.k1 = -2.081261929715610e-02; c.k2 = 0.22600748319395; c.k3 = 5.03580947213895e-1;
        c.k4 = 0.51723167208978; c.k5 = -6.518979800418380e-12;
        break;
    }
    return c;
}

// Blocks of the IEEE-division recompute launch of the reference-rounding form.
constexpr unsigned kRecomputeBlocks = 64;

// Tiles a y/z-sweep block marches through (sweep_tiles): as many as keep at
// least kMarchMinBlocks blocks in the launch, at most HOWMHD_MARCH_STEPS.
#ifndef HOWMHD_MARCH_STEPS
#define HOWMHD_MARCH_STEPS 8
#endif
constexpr unsigned kMarchMinBlocks = 2048;
inline int march_steps(const dim3& tiles) {
    const unsigned long long n = (unsigned long long)tiles.x * tiles.y;
    unsigned long long s = n / kMarchMinBlocks;
    if (s > HOWMHD_MARCH_STEPS) s = HOWMHD_MARCH_STEPS;
    if (s > tiles.y) s = tiles.y;
    return s < 1 ? 1 : (int)s;
}

// Planes per block of the kernels that march through z (k_emf_march,
// k_faces_march).  A block's time is a start (the EMF's first two planes come
// from memory with 24 loads a cell) plus about 1.2 us per plane, so a grid
// that cannot fill the chip with long marches takes as many planes as leave
// kPlaneMarchBlocks blocks, two per CU.  Measured in FP64 against 32 planes
// everywhere: 32^3 EMF 47 -> 10 us and faces 44 -> 7 us (1 plane), 64^3
// 49 -> 20 and 46 -> 11 (3 and 2), 97x75x61 50 -> 24 and 52 -> 23 (4 and 5),
// 128^3 85 -> 74 and 59 -> 53 (17 and 6).  Longer marches than the maxima gain
// nothing: EMF 354 us with 32 or 64 planes at 256^3 (370 with 12); faces
// 333 us with 6 or 32 there, but 147 against 169 us at 192^3, where 32 planes
// make 864 blocks, one more than a round of the 768 the chip holds.
constexpr unsigned kPlaneMarchBlocks = 512;
constexpr int kEmfMaxPlanes = 32, kFaceMaxPlanes = 6;
inline int march_planes(const dim3& tiles, int nz, int most) {
    const unsigned long long n = (unsigned long long)tiles.x * tiles.y * (unsigned)nz;
    const unsigned long long cz = (n + kPlaneMarchBlocks - 1) / kPlaneMarchBlocks;
    return (int)std::min<unsigned long long>(cz, (unsigned long long)most);
}

// The sweeps' blocks in launches of at most kLaunchBlocks.  The runtime refuses
// 2^32 threads along x, which 1-D launches of 256 reach at 2^24 blocks: routed
// tiles are not packed, so a plane of 1 x 8192 x 8192 cells has as many.  (A
// multiple of 8 keeps the launch's blocks on the XCDs that the tile order means.)
// A later launch counts its blocks from 0 again and finds the axes' first blocks
// below them: a block number to add was one more wait at the start of every
// block (routed FP32 steps of 512^2 248.3 -> 249.4 us).
constexpr unsigned kLaunchBlocks = 1u << 23;
template <typename R, typename F>
void launch_parts(const SweepArgs<R>& a, unsigned blocks, const F& launch) {
    SweepArgs<R> part = a;
    for (unsigned done = 0; done < blocks; done += kLaunchBlocks) {
        for (int k = 0; k < 3; ++k) part.ax[k].first = a.ax[k].first - (int)done;
        launch(part, std::min(blocks - done, kLaunchBlocks));
    }
}

// Whether the plain reference-rounding sweeps of a stage run as k_sweep_split.
// With b blocks on a CU a stage of it takes about 4.6 b - 1 us, and one of
// k_sweep, whose blocks have up to four times the interfaces, 6.4 b + 6.6 us.  The
// two are level at 3 blocks of it on a CU beside 1 of k_sweep.  Measured per step,
// k_sweep / split, us: 2 beside 1, orszag_tang 100^2 144 / 124, 128^2 136 / 121;
// 16^3 177 / 155, a line of 30,000 cells 112 / 94; 3 beside 1, 136^2 140 / 147,
// 144^2 139 / 146, 20^3 184 / 179, 16 x 600 184 / 176, a line of 40,001 118 / 119;
// more, 160^2 141 / 160, 24^3 189 / 200, 32^3 218 / 273, a line of 60,000 120 / 132.
// (14^3, 15^3 and 18^3 take 240 us in k_sweep: the last group of columns has 1 or
// 4 of its 32, and a wavefront with so few active lanes is slower.)
constexpr unsigned kCUs = 256;
inline bool split_sweep(const howmhd_gpu_ctx* c) {
    if (c->march_force > 0) return false;
    unsigned long long ns = 0, nk = 0;
    auto per_cu = [](unsigned long long n) { return (n + kCUs - 1) / kCUs; };
    for (int d = 0; d < 3; ++d) {
        if (c->g.n[d] == 1) continue;
        const dim3 t = split_grid(c->g, d), k = sweep_grid(c->g, d, c->xlanes, true);
        ns += (unsigned long long)t.x * t.y;
        nk += (unsigned long long)k.x * k.y;
    }
    return ns <= kLaunchBlocks && 46 * per_cu(ns) < 64 * per_cu(nk) + 71;
}

// Arguments of stage iw's sweeps of the axes in `mask` (bit d: axis d) from qsrc;
// *blocks receives the blocks of the launch.
template <typename R, int MODE>
SweepArgs<R> sweep_args(howmhd_gpu_ctx* c, int iw, const double* qsrc, unsigned mask, unsigned* blocks,
                        bool split = false) {
    SweepArgs<R> a{};
    a.q = qsrc;
    a.g = c->g;
    a.ph = c->ph;
    a.gc = c->gc;
    a.ct_active = c->ctf.active;
    a.mlp = c->mlp;
    a.stats = c->route_now ? c->iwave + (size_t)(iw - 1) * c->nwave : nullptr;
    a.fix = c->fixflag;
    a.fixlist = c->fixlist;
    a.fixctl = c->fixctl;
    a.fixhost = c->fixhost;
    const long long nx = c->g.n[0], ny = c->g.n[1];
    const int order[3] = {1, 2, 0};
    constexpr bool packed = MODE != SW_ROUTED;
    unsigned nb = 0;
    for (int k = 0; k < 3; ++k) {
        const int d = order[k];
        SweepAxis<R>& x = a.ax[k];
        x.dF = (R*)c->dF[d];
        // x: fsy, fsz; y: gsz, gsx; z: hsx, hsy
        x.ct_a = (R*)c->ct[d == 1 ? 3 : 2 * d];
        x.ct_b = (R*)c->ct[d == 1 ? 2 : 2 * d + 1];
        for (int m = 0; m < 8; ++m) x.qoff[m] = (long long)sweep_perm(d, m) * c->g.ncell;
        x.n = c->g.n[d];
        x.per = c->g.per[d];
        const long long nif = x.n + 1 - (x.per ? 1 : 0);  // computed interfaces per line
        const int W = !packed ? 64 : split ? SweepTile<ALONG_X_64>::THREADS : c->xlanes;
        const Lines l = sweep_lines(c->g, d, packed, d == 0 ? SweepTile<ALONG_X>::THREADS / W : SweepTile<ACROSS_X>::LANES);
        x.in = (int)l.in;
        x.nc = (int)(l.period * l.out);
        x.by_o = launch_div((unsigned)l.period);
        x.rows_o = (unsigned)l.in;
        x.sA = (unsigned)(d == 0 ? 1 : d == 1 ? nx : nx * ny);
        x.sB = (unsigned)(d == 2 ? nx : nx * ny);
        x.cF = (long long)c->ncell / x.n * (x.n + 1);
        x.tF = x.sA;
        x.oF = (unsigned)(d == 2 ? nx : nx * (ny + 1));
        x.sS = (unsigned)(d == 0 ? nif : x.sA);
        x.oS = (unsigned)(d == 2 ? nx : nx * nif);
        const dim3 gr = split ? split_grid(c->g, d) : sweep_grid(c->g, d, W, packed);
        x.gx = gr.x; x.gy = gr.y;
        if (d == 0) {
            x.W = W;
            x.rows = split ? 1 : SweepTile<ALONG_X>::THREADS / W;
            x.by_w = launch_div(W);
            x.by_w5 = launch_div(W + 5);
        }
        x.first = (int)nb;
        x.march = 1;
        x.tile0 = c->tile0[d];
        if (d != 0 && sweep_marches<R, MODE>() && !split)
            x.march = c->march_force > 0 ? (int)std::min<unsigned>(c->march_force, gr.y) : march_steps(gr);
        x.by_gx = launch_div(gr.x);
        const unsigned along = (gr.y + x.march - 1) / x.march;
        const unsigned chunk = d == 0 ? gr.x : std::min(gr.x, blocks_for(nx, SweepTile<ACROSS_X>::LANES));
        x.by_chunk = launch_div(chunk);
        x.by_blocks = launch_div(along);
        if (mask & (1u << d)) nb += split ? gr.x * gr.y : blocks_for(gr.x, chunk) * chunk * along;
    }
    *blocks = nb;
    return a;
}

// LDS of a launch of k_sweep: a tile's, of the larger shape that it holds.  With
// the x tile's alone a CU has room for another block where those are not full:
// on lines of cells in the routed sweep, whose tiles are not packed.
template <typename R, int MODE>
size_t sweep_lds(const SweepArgs<R>& a) {
    constexpr size_t x = tile_lds_bytes<R, MODE, ALONG_X>(), yz = tile_lds_bytes<R, MODE, ACROSS_X>();
    static_assert(x <= yz, "LDS of both shapes");
    return a.ax[2].first == 0 ? x : yz;  // (no blocks of y and z)
}

// The IEEE-division launch for the tiles that the sweeps before it queued (it
// exits at once when there are none; no counting there).
template <typename R, int MODE>
void launch_recompute(howmhd_gpu_ctx* c, SweepArgs<R>& a) {
    a.stats = nullptr;
    const size_t lds = sweep_lds<R, MODE>(a);
    hipLaunchKernelGGL((k_sweep<R, MODE, EX, DIV_IEEE>), dim3(kRecomputeBlocks), dim3(256), lds, c->stream, a);
}

// The sweeps of the axes in `mask`, one launch (launch_parts).  Reference rounding: the
// sweeps with unscaled WENO divisions, then the launch for the tiles they
// queued (SW_COLLECT: left to the caller, who waits for the sweep anyway).  Plain
// sweeps of single tiles redo such a tile in place: no launch, which took 4 us
// when empty (a step at 32^3 229 -> 213 us, 64^3 719 -> 700, 96^3 2,249 ->
// 2,207), and no queue for a few blocks where many tiles are out of range (a
// 512^2 run that ends in NaN 3.42 -> 0.74 ms).  The march and the routed sweep
// have no registers for it (816 bytes of scratch a thread).
// One launch instead of one per axis: the last round of one axis's blocks,
// the tail of its marches and its empty recompute launch cost 2% of the
// sweeps at 256^3, and on a grid that leaves the chip idle the axes run side
// by side.
template <typename R, int MODE>
void launch_sweep(howmhd_gpu_ctx* c, SweepArgs<R>& a, unsigned blocks) {
    const size_t lds = sweep_lds<R, MODE>(a);
    if constexpr (EX && MODE == SW_PLAIN) {
        if (a.ax[0].march == 1 && a.ax[1].march == 1) {
            launch_parts(a, blocks, [&](const SweepArgs<R>& p, unsigned nb) {
                hipLaunchKernelGGL((k_sweep<R, MODE, EX, DIV_UNSCALED, true>), dim3(nb), dim3(256), lds, c->stream, p);
            });
            return;
        }
    }
    constexpr int DM = EX ? DIV_UNSCALED : DIV_IEEE;
    launch_parts(a, blocks, [&](const SweepArgs<R>& p, unsigned nb) {
        hipLaunchKernelGGL((k_sweep<R, MODE, EX, DM>), dim3(nb), dim3(256), lds, c->stream, p);
    });
    if constexpr (EX && MODE != SW_COLLECT) {
        if (blocks) launch_recompute<R, MODE>(c, a);
    }
}

inline StageCoef stage_coef(const howmhd_gpu_ctx* c, int iw, double dt) {
    const RK k = rk_coeff(iw);
    StageCoef s;
    s.k1 = k.k1;
    s.k3 = k.k3;
    s.c4 = (iw == 5) ? k.k4 / k.k1 : 0.0;
    s.c5 = (iw == 5) ? k.k5 / k.k1 : 0.0;
    s.dtdx = k.k2 * dt / c->p.dx;   // src/ssprk.cpp:1302-1304
    s.dtdy = k.k2 * dt / c->p.dy;
    s.dtdz = k.k2 * dt / c->p.dz;
    s.stage5 = (iw == 5);
    return s;
}

// The stage combination of stage iw (its inputs: q(0), q(iw-1), stage 2 and
// 3 at stage 5, the faces and interface fluxes of stage iw; its output q(iw)).
template <typename R>
CombineArgs<R> combine_args(howmhd_gpu_ctx* c, int iw, double dt) {
    CombineArgs<R> ca{};
    ca.q0 = c->qbuf[c->qid[0]];
    ca.q2 = c->qbuf[c->qid[2]];
    ca.q3 = c->qbuf[c->qid[3]];
    ca.qp = c->qbuf[c->qid[iw - 1]];
    ca.qo = c->qbuf[c->qid[iw]];
    ca.bo = c->fbuf[c->qid[iw]];
    ca.dFx = (const R*)c->dF[0];
    ca.dFy = (const R*)c->dF[1];
    ca.dFz = (const R*)c->dF[2];
    ca.g = c->g;
    ca.f = c->ctf;
    ca.s = stage_coef(c, iw, dt);
    ca.ph = c->ph;
    ca.cfl = (iw == 5) ? c->cflpart : nullptr;
    ca.floors = (iw == 5) ? c->floorpart : nullptr;
    return ca;
}

// The face update of stage iw.
template <typename R>
FaceArgs<R> face_args(howmhd_gpu_ctx* c, int iw, double dt) {
    FaceArgs<R> fa{};
    fa.Ox = (const R*)c->O[0]; fa.Oy = (const R*)c->O[1]; fa.Oz = (const R*)c->O[2];
    fa.b0 = c->fbuf[c->qid[0]];
    fa.b2 = c->fbuf[c->qid[2]];
    fa.b3 = c->fbuf[c->qid[3]];
    fa.bp = c->fbuf[c->qid[iw - 1]];
    fa.bo = c->fbuf[c->qid[iw]];
    fa.g = c->g;
    fa.f = c->ctf;
    fa.s = stage_coef(c, iw, dt);
    return fa;
}

// The sweeps of a stage: one launch, or one per axis while the kernels are
// being timed.
template <typename R>
int launch_sweeps(howmhd_gpu_ctx* c, int iw, const double* qsrc) {
    unsigned all = 0;
    for (int d = 0; d < 3; ++d)
        if (c->g.n[d] > 1) all |= 1u << d;
    auto go = [&](unsigned mask) {
        unsigned nb = 0;
        if (c->route_now) {
            SweepArgs<R> a = sweep_args<R, SW_ROUTED>(c, iw, qsrc, mask, &nb);
            launch_sweep<R, SW_ROUTED>(c, a, nb);
        } else {
            if constexpr (EX) {
                if (split_sweep(c)) {
                    const SweepArgs<R> a = sweep_args<R, SW_PLAIN>(c, iw, qsrc, mask, &nb, true);
                    if (nb) hipLaunchKernelGGL((k_sweep_split<EX>), dim3(nb), dim3(256), 0, c->stream, a);
                    return;
                }
            }
            SweepArgs<R> a = sweep_args<R, SW_PLAIN>(c, iw, qsrc, mask, &nb);
            launch_sweep<R, SW_PLAIN>(c, a, nb);
        }
    };
    if (!c->timing) {
        go(all);
        HCHECK(c, hipGetLastError());
        return HOWMHD_OK;
    }
    for (int d = 0; d < 3; ++d) {
        if (!(all & (1u << d))) continue;
        TimedLaunch tl(c, HOWMHD_K_SWEEP_X + d);
        go(1u << d);
        HCHECK(c, hipGetLastError());
    }
    return HOWMHD_OK;
}

template <typename R>
int launch_stage(howmhd_gpu_ctx* c, int iw, double dt) {
    const double* qp = c->qbuf[c->qid[iw - 1]];
    int rc = launch_sweeps<R>(c, iw, qp);
    if (rc) return rc;

    if (c->plane) {
        PlaneArgs<R> a{face_args<R>(c, iw, dt), combine_args<R>(c, iw, dt), (const R*)c->ct[2], (const R*)c->ct[0]};
        TimedLaunch tl(c, HOWMHD_K_COMBINE);
        hipLaunchKernelGGL((k_plane<R, EX>), plane_grid(c->g), dim3(256), 0, c->stream, a);
        HCHECK(c, hipGetLastError());
        return HOWMHD_OK;
    }
    const unsigned nb = blocks_for(c->ncell, 256);
    if (c->ctf.use_x && c->ctf.use_y && c->ctf.use_z) {
        EmfMarchArgs<R> e;
        e.fsy = (const R*)c->ct[0]; e.fsz = (const R*)c->ct[1];
        e.gsx = (const R*)c->ct[2]; e.gsz = (const R*)c->ct[3];
        e.hsx = (const R*)c->ct[4]; e.hsy = (const R*)c->ct[5];
        e.Ox = (R*)c->O[0]; e.Oy = (R*)c->O[1]; e.Oz = (R*)c->O[2];
        e.g = c->g;
        dim3 grid(blocks_for(c->g.n[0], EMF_OX), blocks_for(c->g.n[1], EMF_OY));
        e.cz = march_planes(grid, c->g.n[2], kEmfMaxPlanes);
        grid.z = blocks_for(c->g.n[2], e.cz);
        {
            TimedLaunch tl(c, HOWMHD_K_EMF);
            hipLaunchKernelGGL((k_emf_march<R, EX>), grid, dim3(EMF_THREADS), 0, c->stream, e);
        }
        HCHECK(c, hipGetLastError());
    } else if (c->ctf.active) {
        EmfArgs<R> e;
        e.fsz = (const R*)c->ct[1]; e.gsz = (const R*)c->ct[3];
        e.hsx = (const R*)c->ct[4]; e.hsy = (const R*)c->ct[5];
        e.Oy2 = (R*)c->O2[1]; e.Oz2 = (R*)c->O2[2];
        e.g = c->g;
        e.f = c->ctf;
        {
            TimedLaunch tl(c, HOWMHD_K_EMF2);
            hipLaunchKernelGGL((k_emf2<R, EX>), dim3(nb), dim3(256), 0, c->stream, e);
        }
        HCHECK(c, hipGetLastError());
        SmoothArgs<R> m;
        m.Oy2 = (const R*)c->O2[1]; m.Oz2 = (const R*)c->O2[2];
        m.Oy = (R*)c->O[1]; m.Oz = (R*)c->O[2];
        m.g = c->g;
        m.f = c->ctf;
        {
            TimedLaunch tl(c, HOWMHD_K_EMF);
            hipLaunchKernelGGL((k_emf<R, EX>), dim3(nb), dim3(256), 0, c->stream, m);
        }
        HCHECK(c, hipGetLastError());
    }
    FaceArgs<R> fa = face_args<R>(c, iw, dt);
    if (c->ctf.active) {
        TimedLaunch tl(c, HOWMHD_K_FACES);
        if (c->ctf.use_x && c->ctf.use_y && c->ctf.use_z) {
            dim3 fgrid(blocks_for(c->g.n[0], FACE_TX), blocks_for(c->g.n[1], FACE_TY));
            fa.cz = march_planes(fgrid, c->g.n[2], kFaceMaxPlanes);
            fgrid.z = blocks_for(c->g.n[2], fa.cz);
            hipLaunchKernelGGL((k_faces_march<R, EX>), fgrid, dim3(256), 0, c->stream, fa);
        } else {
            const dim3 fgrid(blocks_for(c->g.n[0], FACE_TX), blocks_for(c->g.n[1], FACE_TY), c->g.n[2]);
            hipLaunchKernelGGL((k_faces<R, EX>), fgrid, dim3(256), 0, c->stream, fa);
        }
    }
    HCHECK(c, hipGetLastError());

    {
        const CombineArgs<R> ca = combine_args<R>(c, iw, dt);
        TimedLaunch tl(c, HOWMHD_K_COMBINE);
        if (c->ctf.active)
            hipLaunchKernelGGL((k_combine<R, EX, false>), dim3(nb), dim3(256), 0, c->stream, ca, fa);
        else
            hipLaunchKernelGGL((k_combine<R, EX, true>), dim3(nb), dim3(256), 0, c->stream, ca, fa);
    }
    HCHECK(c, hipGetLastError());
    return HOWMHD_OK;
}

}  // namespace
}  // namespace howmhd
