"""Host transfers where they are cut into chunks (needs a GPU): several
variables to a chunk, ranges of y planes with a remainder, ranges of x of one
y plane, axes so short that a cell has several ghost images, and a caller's
array in device memory.  Every value, ghosts included, is compared bit for bit
with numpy index maps.
"""
import ctypes as C

import numpy as np
import pytest

import howmhd as H
from test_gpu_transfer import OPEN, PER, _expected, _params

pytestmark = pytest.mark.gpu

SHAPES = [
    ((3, 4, 5), (PER, OPEN, PER)),         # one chunk; three to five cells an axis
    ((4, 3, 3), (OPEN, PER, OPEN)),
    ((33, 65, 31), (PER, PER, OPEN)),      # two variables' worth of slots, ragged tiles
    ((97, 75, 61), (OPEN, OPEN, OPEN)),    # y ranges with a remainder
    ((700, 3, 500), (PER, OPEN, OPEN)),    # a y plane larger than a slot: x ranges
    ((3, 400, 300), (OPEN, PER, PER)),
    ((1, 5, 40000), (PER, PER, OPEN)),
]


@pytest.mark.parametrize("shape,bc", SHAPES, ids=["x".join(map(str, s)) for s, _ in SHAPES])
def test_transfer_chunks(shape, bc, require_gpu):
    print(f"[transfer chunks] shape={shape} bc={bc}", flush=True)
    rng = np.random.default_rng(sum(shape))
    full = tuple(n + 6 for n in shape)
    with H.GpuSolver(_params(*shape, bc)) as g:
        q, b = rng.standard_normal((8,) + full), rng.standard_normal((3,) + full)
        for _ in range(2):  # the second pass reuses every slot
            g.upload_q0(q)
            g.upload_faces(b)
            for got, src in ((g.q0(), q), (g.faces(), b)):
                assert np.array_equal(got.view(np.int64), _expected(src, shape, bc).view(np.int64))
            q, b = q[::-1].copy(), b[::-1].copy()


def test_transfer_device_pointer(require_gpu):
    """The calls take host arrays; a device pointer is copied too."""
    import torch

    shape, bc = (20, 9, 11), (PER, OPEN, PER)
    q = torch.randn((8,) + tuple(n + 6 for n in shape), dtype=torch.float64, device="cuda")
    out = torch.zeros_like(q)
    torch.cuda.synchronize()
    dp = lambda t: C.cast(t.data_ptr(), C.POINTER(C.c_double))  # noqa: E731
    with H.GpuSolver(_params(*shape, bc)) as g:
        assert g.lib.howmhd_gpu_upload_q0(g.h, dp(q)) == 0
        assert g.lib.howmhd_gpu_download_q0(g.h, dp(out)) == 0
    assert np.array_equal(out.cpu().numpy(), _expected(q.cpu().numpy(), shape, bc))
