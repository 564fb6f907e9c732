"""The MLP's products at the edges of their tiles: rows, widths and outputs that
are no multiples of 32 or 128, a K of one, K below and above a wave's share,
rows of operands that are not 16-byte aligned, and sizes on either side of the
line between the two kernels, in forward and gradient, against the FP64 oracle
on the same BF16-rounded operands.  Bars: those of the MLP test in
tests/test_engine_gpu.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,width,depth,n_out,rows", [
    (1, 8, 1, 1, 1), (5, 33, 2, 17, 31), (3, 64, 3, 65, 129), (7, 130, 1, 257, 300),
    (5, 256, 2, 300, 33),
    (3, 33, 1, 1030, 4100),     # large forward products of odd K
    (2, 1157, 1, 2931, 37),     # a large weight gradient, K = 37 rows
    (2, 1030, 2, 19, 4100)])    # large products with K = 1030, all three kinds
def test_product_edges(pkg, n_in, width, depth, n_out, rows):
    from oracle import mlp_oracle as mo
    rng = np.random.default_rng(width + rows)
    with pkg.engine.Context(0) as ctx, \
            pkg.engine.Mlp(ctx, n_in, width, depth, n_out, seed=3) as net:
        shapes = mo.layer_shapes(n_in, width, depth, n_out)
        p = net.params().astype(np.float64)
        x = rng.normal(size=(rows, n_in)).astype(np.float32)
        t = rng.normal(size=(rows, n_out)).astype(np.float32)
        y = net.forward(x)
        loss, g = net.gradient(x, t)
    y_o, _ = mo.forward(p, shapes, x, bf=True)
    loss_o, g_o = mo.loss_and_grad(p, shapes, x, t, bf=True)
    ey = np.linalg.norm(y - y_o) / np.linalg.norm(y_o)
    eg = np.linalg.norm(g - g_o) / np.linalg.norm(g_o)
    print("forward rel L2 %.2e; loss %.6e vs %.6e; gradient rel L2 %.2e" % (ey, loss, loss_o, eg))
    assert ey < 1e-3
    assert abs(loss - loss_o) < 1e-4 * loss_o
    assert eg < 2e-3
