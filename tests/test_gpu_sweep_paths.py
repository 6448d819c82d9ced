"""The reference-rounding sweeps of the smallest grids run split over the
wavefronts of a block, the others as single tiles (1) or as marches that queue
tiles for an IEEE-division launch (2) (needs a GPU).  Every parity case is small
enough for the split sweep; here the same cases run on the others
(HOWMHD_SWEEP_MARCH), bit for bit against the CPU restatement: the case list,
operands beyond the unscaled divisions, subnormal squares, a cell without
positive density, and one cell along x.  And a grid on each side of the rule.
"""
import pytest

import howmhd as H
import mlp_oracle as M
import oracle_ctypes as O
import test_gpu_parity as P
from test_gpu_launch_rules import _step_matches

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["1", "2"])
def tiles(request, monkeypatch):
    monkeypatch.setenv("HOWMHD_SWEEP_MARCH", request.param)
    print(f"[sweep paths] {request.param} tiles a block", flush=True)


@pytest.mark.parametrize("case", list(P.CASES))
def test_tiles_on_parity_cases(case, tiles, require_gpu):
    P.test_fp64_bitwise(case, require_gpu)


@pytest.mark.parametrize("problem,kw", [("mhd_blast3d", dict(nx=16, ny=16, nz=16)),
                                        ("orszag_tang", dict(nx=32, ny=32, nz=1, cour=0.8))])
def test_tiles_recompute(problem, kw, tiles, require_gpu):
    P.test_fp64_bitwise_large_weno_operands(problem, kw, require_gpu)
    P.test_fp64_bitwise_small_sqrt_operands(problem, kw, require_gpu)
    P.test_fp64_bitwise_nonpositive_density_cell(-0.25, require_gpu)
    P.test_fp64_bitwise_nonpositive_density_cell(1e-300, require_gpu)
    P.test_fp64_bitwise_degenerate_x("mpi_smooth3d", dict(nx=1, ny=12, nz=10), require_gpu)


# grids on both sides of the rule (512 blocks of the split sweep and one row
# more), a line longer than 512 blocks, thin grids; interfaces that fill the 64
# of a block and one more, last columns of 1 to 15
@pytest.mark.parametrize("n,bc", [((256, 128, 1), "periodic"), ((256, 130, 1), "periodic"), ((65, 17, 17), "open"),
                                  ((64, 20, 18), "open"), ((63, 5, 3), "open"), ((64, 16, 1), "periodic"),
                                  ((65, 17, 1), "open"), ((128, 128, 1), "open"), ((128, 132, 1), "periodic"),
                                  ((40001, 1, 1), "open"), ((4100, 3, 1), "periodic"), ((3, 1, 2050), "periodic")])
def test_split_rule(n, bc, require_gpu):
    _step_matches("mpi_smooth3d", n, bc, steps=2)


@pytest.mark.parametrize("n,bc", [((16, 16, 16), "periodic"), ((33, 17, 15), "open")])
def test_labels_beyond_the_unscaled_range(n, bc, require_gpu):
    """Samples of a flow scaled as in the large-operand parity test, whose tiles
    go through the IEEE-division launch, and of the flow itself afterwards on
    the same solver, whose tiles do not: labels of both match the restatement."""
    torch = pytest.importorskip("torch")
    run = H.parse(H.make_input(problem="mhd_blast3d", nx=n[0], ny=n[1], nz=n[2], nt=1,
                               tend=1.0, x1bc=bc, x2bc=bc, x3bc=bc))
    p, q0 = H.gpu_params(run), H.init_problem(run)
    big = q0.copy()
    big[[0, 1, 2, 3, 7]] *= 1e50
    big[[4, 5, 6]] *= 1e25
    print(f"[sweep paths] labels {n} {bc}", flush=True)
    with H.GpuSolver(p) as g:
        for q, scaled in ((big, True), (q0, False), (big, True)):
            g.upload_q0(q)
            g.init_faces()
            O.large_t_count(reset=True)
            for d in range(3):
                X = torch.empty((g.n_samples(d), H.MLP_NFEAT), dtype=torch.float32, device="cuda")
                y = torch.empty(g.n_samples(d), dtype=torch.float32, device="cuda")
                g.collect_samples(d, X, y)
                lab, dev = M.interface_labels(H.active(g.q0()), d, p.bc[d] == H.BC["periodic"], p.gam, O.line_maxdev,
                                              p.rhomin, p.pgmin)
                clear = abs(dev - 0.05) > 1e-9
                assert (y.cpu().numpy() == lab)[clear].all()
            assert (O.large_t_count() > 0) == scaled


# rows and columns numbered through both transverse axes, x tiles of 16 to 256
# interfaces a row: rows shorter than the least, one more and less than 16, 48, 64
# and 256, tiles that span several planes, a last tile of one line
@pytest.mark.parametrize("n,bc", [((5, 37, 11), "open"), ((17, 9, 16), "periodic"), ((47, 5, 13), "open"),
                                  ((65, 3, 17), "periodic"), ((72, 11, 7), "open"), ((255, 3, 5), "open"),
                                  ((257, 4, 3), "periodic"), ((33, 1, 65), "open"), ((300, 1, 1), "open")])
def test_packed_lines(n, bc, tiles, require_gpu):
    _step_matches("mpi_smooth3d", n, bc, steps=1)


# the largest grids of the split sweep beside the smallest of k_sweep (64 interfaces
# a block, 256 CUs: 512 blocks and more; one row, column or line of cells apart
# where the packed tiles allow it), for every set of axes; True: split.  The CPU
# test of the launches checks the sides.
SPLIT_EDGE = [((32768, 1, 1), "periodic", True), ((32769, 1, 1), "periodic", False),
              ((32767, 1, 1), "open", True), ((32768, 1, 1), "open", False),
              ((128, 128, 1), "periodic", True), ((128, 129, 1), "periodic", False),
              ((127, 120, 1), "open", True), ((127, 128, 1), "open", False),
              ((8192, 3, 1), "periodic", True), ((12000, 3, 1), "open", False),
              ((128, 1, 128), "periodic", True), ((129, 1, 128), "periodic", False),
              ((1, 127, 127), "open", True), ((1, 128, 132), "periodic", False),
              ((17, 17, 17), "open", True), ((18, 18, 18), "periodic", False),
              ((64, 16, 9), "periodic", True), ((65, 16, 9), "periodic", False)]


@pytest.mark.parametrize("n,bc,split", SPLIT_EDGE)
def test_split_edge(n, bc, split, require_gpu):
    # (grids without an x axis end in NaN, whose sign bits are the processor's, in the second step)
    _step_matches("mpi_smooth3d", n, bc, steps=2 if n[0] > 1 else 1)
