"""Inference and gradient of the indicator network at the edges of their tiles
(needs a GPU): one sample, one less and one more than a 16-sample tile, a
64-sample group and the samples of a 128-sample block, a batch beyond the
largest launch of either kernel, and features that are only 4-byte aligned.

Tolerances: an activation that rounds to the other bf16 neighbour moves by
2^-8 of itself and passes two layers; 5 x 2^-8 covers every activation of a
sample doing so at once.  The loss is a mean of logits' errors, each at most
that bound.
"""
import numpy as np
import pytest

import howmhd as H
import mlp_oracle as M

pytestmark = pytest.mark.gpu

TOL = 5 * 2.0 ** -8


@pytest.mark.parametrize("n,shift", [(1, 0), (15, 1), (16, 0), (17, 1), (63, 0), (64, 1), (65, 0), (127, 0), (128, 1),
                                     (129, 0), (32768 + 5, 1), (524288 + 17, 0)])
def test_mlp_tiles(n, shift, require_gpu):
    import torch

    print(f"[mlp tiles] n={n} shift={shift}", flush=True)
    rng = np.random.default_rng(n)
    X = rng.uniform(0, 1, (n, 18)).astype(np.float32)
    y = (rng.uniform(size=n) < 0.4).astype(np.float32)
    P = M.init_params(4)
    P[M.OFF_B1:M.OFF_W2] = rng.normal(0, 0.2, 32)
    P[M.OFF_B2:M.OFF_W3] = rng.normal(0, 0.2, 32)
    # NaN around the samples: a sample beyond the last must not count
    flat = torch.full((18 * n + 64 * 18 + 1,), float("nan"), device="cuda")
    flat[shift:shift + 18 * n] = torch.from_numpy(X.reshape(-1)).cuda()
    Xd = flat[shift:shift + 18 * n].view(n, 18)
    yd = torch.from_numpy(y).cuda()
    Pd = torch.from_numpy(P).cuda()
    z = H.mlp_infer(Xd, Pd).cpu().numpy()
    zr, _ = M.forward(P, X)
    assert np.all(np.abs(z - zr) <= TOL * (1 + np.abs(zr)))
    G0 = rng.normal(0, 1e-3, M.NPARAM).astype(np.float32)  # the gradient is added to what is there
    G, loss = H.mlp_grad(Xd, yd, Pd, pos_weight=2.5, scale=1.0 / n, G=torch.from_numpy(G0).cuda())
    lr, Gr = M.loss_and_grad(P, X, y, pos_weight=2.5, scale=1.0 / n)
    assert abs(float(loss.cpu()) - lr) <= TOL * (1 + abs(lr))
    G = G.cpu().numpy().astype(np.float64) - G0
    for a, b in ((0, M.OFF_B1), (M.OFF_B1, M.OFF_W2), (M.OFF_W2, M.OFF_B2), (M.OFF_B2, M.OFF_W3),
                 (M.OFF_W3, M.OFF_B3), (M.OFF_B3, M.NPARAM)):
        assert np.linalg.norm(G[a:b] - Gr[a:b]) <= TOL * np.linalg.norm(Gr[a:b]) + 1e-7, (a, b)
