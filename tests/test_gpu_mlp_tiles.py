"""The network's products at the edges of their tiles: one row and one unit,
widths and batches with a remainder in every tile, and a batch large enough for
the wide tiles.  One hidden layer on dyadic data (exact sums) forward bit for
bit, gradients to FP32 accumulation order; after an Adam step the weights the
products read are the parameters handed out."""
import numpy as np
import pytest

import fedg
import fedg_oracle_mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,B", [((1, 1, 1, 1), 1), ((33, 40, 1, 17), 33), ((20, 24, 1, 4), 95), ((47, 31, 3, 65), 130),
                                    ((64, 256, 1, 256), 8224)])
def test_tiles(dims, B):
    print(f"mlp tiles {dims} B={B}", flush=True)
    lay = M.Layout(*dims)
    rng = np.random.default_rng(B)
    pick = lambda n, v: rng.choice(np.asarray(v, dtype=np.float32), size=n)  # noqa: E731
    p = pick(lay.nparam, [-1.0, -0.5, 0.0, 0.5, 1.0])
    for l in range(lay.nl):
        p[lay.boff[l]:lay.boff[l] + lay.dims[l + 1]] = pick(lay.dims[l + 1], [-0.25, 0.0, 0.25])
    X = pick((B, dims[0]), [-1.0, -0.75, -0.5, -0.25, 0.0, 0.25, 0.5, 0.75, 1.0])
    net = fedg.Mlp(*dims)
    net.set_params(p)

    def forward():
        dX, dY = fedg.DevField32(X.size, X), fedg.DevField32(B * dims[3])
        net.forward(dX, dY, B)
        return dY.download().reshape(B, dims[3])

    Y, Yo = forward(), M.forward(lay, p, X, rnd=True)[-1]
    if dims[2] == 1:
        assert np.array_equal(Y, Yo)
    else:
        assert np.linalg.norm(Y - Yo) <= 1e-4 * np.linalg.norm(Yo)
    T = (Yo + rng.integers(-2, 3, Yo.shape)).astype(np.float32)
    T.flat[0] += 1.0
    dX, dT = fedg.DevField32(X.size, X), fedg.DevField32(T.size, T)
    loss = net.loss_grad(dX, dT, B)
    lo, go = M.loss_grad(lay, p, X, T, rnd=True)
    assert loss == pytest.approx(lo, rel=1e-4)
    g = net.grads()
    for l in range(lay.nl):
        w = slice(lay.woff[l], lay.woff[l] + lay.dims[l] * lay.dims[l + 1])
        b = slice(lay.boff[l], lay.boff[l] + lay.dims[l + 1])
        for s in (w, b):
            assert np.linalg.norm(g[s] - go[s]) <= 2e-3 * np.linalg.norm(go[s]), f"layer {l}"
    net.adam_step(1e-2)
    after = forward()
    assert not np.array_equal(after, Y)
    net.set_params(net.params())
    assert np.array_equal(after, forward())
    net.close()
