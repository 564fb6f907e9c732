"""Work items of the incoherent sum: many short orientations stay whole (a segment
each costs more in the reduction than it saves, and up to 8 GiB of partial
grids), a long one among few is cut; both against the FP64 oracle (bar of the
path, 1e-10), and items that hold many orientations."""
import numpy as np
import pytest

import metrics as M
from conftest import load_fixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts, cells, items", [
    ([20] * 200, (91, 16), "whole"), ([1, 0, 3] * 400, (7, 5), "whole"),
    ([300], (13, 5), "cut"), ([15, 64, 3, 0] + [9] * 12, (31, 12), "cut"),
    ([15, 63, 3, 0] + [9] * 12, (31, 12), "whole")])
def test_items(pkg, oracle, counts, cells, items):
    """The rule's line lies at four beams in the longest orientation for each
    orientation: 64 for 16."""
    abi = pkg.abi
    fx = load_fixture("sobol_average")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    batch = pkg.synthetic.resample(src, np.asarray(counts), seed=len(counts))
    grid = abi.Grid.build(np.linspace(0.05, 3.1, cells[0]), cells[1])
    with pkg.engine.Context(0) as ctx:
        ctx.set_timing(True)
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        for target in (65536, 300):
            ctx.set_target_blocks(target)
            m = ctx.mueller(abi.PREC_FP64 | abi.INCOHERENT)[0]
            n = ctx.timing()["n_items"]
            if items == "whole":
                assert n <= len(counts)
            elif target == 65536:
                assert n > len(counts)
            e = M.grid_l2(m, oracle.incoherent(grid, batch, consts), grid.theta)
            assert e < 1e-10
