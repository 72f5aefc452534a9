"""Weight, bias and input gradients of the Schur-stencil network around the line between one
workgroup per output pair (8,192 points) and partial sums over chunks of points, against the
float64 oracle: every gradient is a sum of at most T = batch x points products rounded to FP32
in runs of at most 64 that are then added in FP64, so its error stays below 70 x 2^-24 = 4e-6 of
the sum of magnitudes; relative to the gradient's norm, with random signs, 2e-5 leaves a factor
of the ratio of the two.  Points whose activation lies within rounding of zero may switch their
ReLU, which the same bound covers at these sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,B,C,Ly", [((16, 16, 16), 2, 8, 2),    # 8,192 points: one chunk
                                         ((19, 16, 27), 1, 16, 1),   # 8,208: chunks, 9 input channels
                                         ((33, 17, 15), 1, 8, 2),    # 8,415: eight channels
                                         ((23, 21, 18), 1, 32, 2),   # channel blocks
                                         ((41, 42, 40), 1, 16, 2)])  # above 65,536: 16-channel blocks
def test_gradients_match_oracle(grid, B, C, Ly):
    from underworld2_amd import learned
    from oracle import nn_oracle as N
    rng = np.random.default_rng(5)
    E = int(np.prod(grid))
    net = learned.StencilNet(C, Ly, seed=2)
    on = N.StencilNet(grid, C, Ly)
    p = net.get_params()
    wo, bo = on.specs[-1][2:4]
    p[wo:] = (0.1 * rng.standard_normal(p.size - wo)).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((B, 9, E)).astype(np.float32)
    r = rng.standard_normal((B, E)).astype(np.float32)
    t = rng.standard_normal((B, E)).astype(np.float32)
    lg, gg = net.loss_grad(grid, x, r, t)
    lo, go, _ = on.loss_grad(p.astype(np.float64), x, r, t)
    err = np.linalg.norm(gg - go) / np.linalg.norm(go)
    print(f"{grid} x {B}, C={C}: gradient error {err:.1e}", flush=True)
    assert abs(lg - lo) < 1e-5 * abs(lo)
    assert err < 2e-5
    l2, g2 = net.loss_grad(grid, x, r, t)
    assert l2 == lg and np.array_equal(g2, gg)
