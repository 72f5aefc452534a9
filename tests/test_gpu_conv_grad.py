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


@pytest.mark.parametrize("grid,B,C", [((6, 5, 4), 2, 8), ((23, 20, 19), 1, 8)])  # one chunk, several
def test_infinite_features_of_inactive_channels(grid, B, C):
    """An infinite feature whose weights are negative only reaches inactive channels: their gradients
    are zero there, and a product of the two is left out of the sums instead of making them NaN.  The
    gradients are those for a large finite feature, which the same ReLUs drop, bit for bit."""
    from underworld2_amd import learned
    rng = np.random.default_rng(7)
    E = int(np.prod(grid))
    net = learned.StencilNet(C, 1, seed=4)
    p = net.get_params()
    w = p[:C * 9 * 27].reshape(C, 9, 27)
    w[:, 2] = -np.abs(w[:, 2]) - 0.01
    net.set_params(p)
    x = rng.standard_normal((B, 9, E)).astype(np.float32)
    r, t = (rng.standard_normal((B, E)).astype(np.float32) for _ in range(2))
    out = []
    for v in (np.inf, 1e30):
        x[:, 2, E // 2] = v
        out.append(net.loss_grad(grid, x, r, t))
    assert np.isfinite(out[0][0]) and np.isfinite(out[0][1]).all()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
