"""Launch rules that depend on the grid size, against the CPU restatement bit
for bit (needs a GPU; plain FP64, one step, q and faces).

z-marching EMF and face kernels: planes per block from one (a grid far too
small for the chip) over a few, with and without a remainder, to a last chunk
of one plane; periodic and open edges.
"""
import numpy as np
import pytest

import howmhd as H
import oracle_ctypes as O

pytestmark = pytest.mark.gpu


def _bits(a, one_nan):
    a = np.where(np.isnan(a), np.nan, a) if one_nan else a
    return a.view(np.int64)


def _step_matches(problem, n, bc, steps=1, one_nan=False):
    run = H.parse(H.make_input(problem=problem, nx=n[0], ny=n[1], nz=n[2], nt=1, tend=1.0, x1bc=bc, x2bc=bc, x3bc=bc))
    print(f"[launch rules] {problem} {n} {bc}", flush=True)
    p, q0 = H.gpu_params(run), H.init_problem(run)
    ref, gpu = O.RefSolver(p), H.GpuSolver(p)
    for s in (ref, gpu):
        s.upload_q0(q0)
        s.init_faces()
    for _ in range(steps):
        dt = ref.tstep()
        assert gpu.tstep() == dt
        ref.ssprk(dt)
        gpu.ssprk(dt)
    for a, b in ((gpu.q0(), ref.q0()), (gpu.faces(), ref.faces())):
        assert np.array_equal(_bits(H.active(a), one_nan), _bits(H.active(b), one_nan))
    gpu.close()
    ref.close()


# (EMF planes per block, face planes): (1, 1) with 5 planes; (2, 2) with an odd
# depth; (3, 2), last EMF chunk one plane; (5, 5), last chunks 4 and 4; (1, 6)
@pytest.mark.parametrize("n,bc", [((33, 30, 5), "open"), ((70, 64, 41), "periodic"), ((64, 50, 67), "open"),
                                  ((130, 61, 64), "periodic"), ((9, 8, 400), "open")])
def test_planes_per_block(n, bc, require_gpu):
    _step_matches("mpi_smooth3d", n, bc)


# the axes' blocks in one launch: an axis of one cell in each place, ragged
# tiles on every axis, more rows than a group of 8 in x, marches (the sweeps of
# the last grid march through 2 tiles)
@pytest.mark.parametrize("n,bc", [((67, 1, 35), "open"), ((70, 41, 1), "periodic"), ((200, 1, 1), "open"),
                                  ((65, 35, 9), "open"), ((97, 120, 130), "periodic")])
def test_axes_in_one_launch(n, bc, require_gpu):
    _step_matches("mpi_smooth3d", n, bc)


def test_timed_launches_change_no_bit(require_gpu):
    """Timing launches the axes one by one and reports each."""
    run = H.parse(H.make_input(problem="mhd_blast3d", nx=40, ny=33, nz=20, nt=1, tend=1.0))
    p, q0 = H.gpu_params(run), H.init_problem(run)
    out = []
    for timed in (False, True):
        with H.GpuSolver(p) as g:
            g.upload_q0(q0)
            g.init_faces()
            g.set_timing(timed)
            for _ in range(2):
                g.ssprk(g.tstep())
            if timed:
                assert [g.timing()[k][1] for k in ("sweep_x", "sweep_y", "sweep_z")] == [10, 10, 10]
            out.append(g.q0())
    assert np.array_equal(out[0].view(np.int64), out[1].view(np.int64))


# CFL maxima folded by one block (at most 512 partials) and by several, from
# q(0) after the upload and from the step's own maxima
@pytest.mark.parametrize("n", [(131072, 1, 1), (131073, 1, 1), (700, 800, 1)])
def test_cfl_fold(n, require_gpu):
    _step_matches("mpi_smooth3d", n, "periodic", steps=2)


def test_counts_fold_over_blocks(require_gpu):
    """Routed counts over more tiles than one block folds, in both counting
    modes: every interface is counted once per sweep and stage."""
    run = H.parse(H.make_input(problem="mhd_blast3d", nx=72, ny=64, nz=70, nt=1, tend=1.0))
    q0 = H.init_problem(run)
    P, thr = H.load_indicator(H.PKG_DIR / "weights" / "indicator_mlp.txt")
    seen = []
    for mode in (1, 2):
        with H.GpuSolver(H.gpu_params(run)) as g:
            g.set_indicator(P, thr, enable=mode)
            g.upload_q0(q0)
            g.init_faces()
            for _ in range(3):
                g.ssprk(g.tstep())
            st = g.indicator_stats()
            assert st["total"] == 3 * 5 * 3 * 72 * 64 * 70 and 0 < st["flagged"] < st["total"]
            assert 0.0 < g.diag().flagged_fraction < 1.0
            seen.append((st["flagged"], st["waves_flagged"], st["waves_total"], g.diag().flagged_fraction))
            assert g.indicator_stats()["total"] == 0
    assert seen[0] == seen[1]


# one-plane grids: everything after the sweeps in one launch of 32 x 8 tiles.
# Axes shorter than the halos (3 to 5 cells), one cell more and less than a
# tile, a last tile of one column or row, both boundaries
@pytest.mark.parametrize("n", [(3, 3, 1), (5, 4, 1), (31, 7, 1), (32, 8, 1), (33, 9, 1), (64, 17, 1), (130, 77, 1)])
@pytest.mark.parametrize("bc", ["periodic", "open"])
def test_one_plane(n, bc, require_gpu):
    _step_matches("mpi_smooth3d", n, bc, steps=2)


# grids of one axis (no EMF): the combination carries the faces.  One cell less
# and more than a block, each axis, both boundaries.  On a y or z line the old
# stages have no weights (the x update applies them), and the second step of an
# open one ends in NaN at the same cells on both sides, whose sign bits are the
# processor's own.
@pytest.mark.parametrize("n", [(3, 1, 1), (255, 1, 1), (257, 1, 1), (1, 256, 1), (1, 1, 600)])
@pytest.mark.parametrize("bc", ["periodic", "open"])
def test_one_axis(n, bc, require_gpu):
    _step_matches("mpi_smooth3d", n, bc, steps=2, one_nan=True)


# arrays of a context in FP64, values a cell: q and faces of 5 stages, 7 fluxes an
# axis, 6 CT terms; the EMF and the unsmoothed one of two-axis grids that k_plane
# does not take.  Beside them, at most `more`: arrays of a few values a tile (88 B a
# tile of the sweeps, which has 8 cells on a y-z grid: 2.8 values a cell), the
# last interfaces, allocations rounded up to 2 MiB.
@pytest.mark.parametrize("n,values,more", [((4096, 4000, 1), 40 + 15 + 14 + 6, 1.0),
                                           ((16000000, 1, 1), 40 + 15 + 7 + 6, 1.0),
                                           ((4096, 1, 4000), 40 + 15 + 14 + 6 + 2, 1.0),
                                           ((1, 4096, 4000), 40 + 15 + 14 + 6 + 2, 3.5)])
def test_context_memory(n, values, more, require_gpu):
    torch = pytest.importorskip("torch")
    params = H.gpu_params(H.parse(H.make_input(problem="mpi_smooth3d", nx=8, ny=8, nz=8, nt=1, tend=1.0)))
    H.GpuSolver(params).close()  # what the process allocates once
    params.nx, params.ny, params.nz = n
    before = torch.cuda.mem_get_info()[0]
    g = H.GpuSolver(params)
    used = (before - torch.cuda.mem_get_info()[0]) / (8.0 * n[0] * n[1] * n[2])
    g.close()
    print(f"[launch rules] memory {n}: {used:.2f} values a cell", flush=True)
    assert values <= used < values + more
