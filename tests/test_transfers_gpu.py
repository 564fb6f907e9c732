"""Copies through the page-locked chunks (1 MiB, 4 MiB from 8 MiB on, shared by
threads from 512 KiB on): sizes on either side of those lines and off them,
up and down, bit for bit against the same data in small pieces."""
import numpy as np
import pytest

from conftest import load_fixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 181, 182, 1449, 1450, 3000])
def test_result_sizes(pkg, rows):
    """rows x 724 FP32 outputs: up to 525 KB in one chunk, 1449 rows just above
    4 MiB, 3000 rows 8.7 MB, against the rows one chunk at a time."""
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, 5)).astype(np.float32)
    with pkg.engine.Context(0) as ctx, pkg.engine.Mlp(ctx, 5, 32, 2, 724, seed=2) as net:
        y = net.forward(x)
        z = np.concatenate([net.forward(x[i:i + 100]) for i in range(0, rows, 100)])
    np.testing.assert_array_equal(y, z)


@pytest.mark.parametrize("n_beams", [1, 2900, 2920, 23000, 30000])
def test_batch_sizes(pkg, n_beams):
    """Batches of 0.4 KB to 12 MB (1 MiB lies near 2,900 beams of four vertices
    at 352 bytes each, 8 MiB near 23,000), against page-locked staging, which
    goes up in one piece; and accumulation into grids that hold something."""
    abi = pkg.abi
    fx = load_fixture("sobol_average")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    batch = pkg.synthetic.resample(src, np.array([n_beams]), seed=n_beams)
    grid = abi.Grid.build(np.linspace(0.0, np.pi, 257), 33)  # 1.1 MB of results
    out = []
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        for up in (ctx.upload, ctx.upload_staged):
            up(batch, consts)
            ctx.diffract(abi.PREC_MIXED | abi.NOSHADOW)
            a, b = np.full((2, grid.n_az, grid.n_zen + 1, 16), 0.5)
            ctx.accumulate(a, b)
            m, mn = np.zeros_like(a), np.zeros_like(a)
            ctx.accumulate(m, mn)
            np.testing.assert_array_equal(a, 0.5 + m)
            np.testing.assert_array_equal(b, 0.5 + mn)
            out.append((m, mn))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
