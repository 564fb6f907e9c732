"""Beams with a value that is not finite do not count: their aperture integral is
NaN in every direction, and the reference skips such a beam
(src/handler/HandlerPO.cpp:2742).  Every polygon class has some, their Jones
matrices a thousand times the others'."""
import numpy as np
import pytest

from conftest import load_fixture

pytestmark = pytest.mark.gpu


def _batch(abi, beams, src, **changed):
    verts = np.concatenate([np.arange(src.vert_offsets[b], src.vert_offsets[b + 1])
                            for b in beams])
    d = dict(beam_scalars=src.beam_scalars[beams].copy(), vx=src.vx[verts].copy(),
             vy=src.vy[verts].copy())
    vo = np.r_[0, np.cumsum(src.beam_nv[beams])]
    for k, f in changed.items():
        f(d[k], vo)
    return abi.BeamBatch([0, len(beams)], [1.0], d["beam_scalars"], src.beam_nv[beams],
                         np.arange(len(beams)) % 5 == 4, vo, d["vx"], d["vy"],
                         src.slope_yx[verts], src.slope_xy[verts], src.edge_flags[verts])


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("where", ["centre", "vertex", "axis", "direction"])
def test_beams_with_values_not_finite(pkg, where, value):
    """Every third beam spoilt, against the batch without them: the same terms in
    another order, 60 of them: 60 2^-53 and 60 2^-24 of the largest."""
    abi = pkg.abi
    fx = load_fixture("config3_aggregate")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    beams = np.concatenate([np.flatnonzero(src.beam_nv == k)[:18] for k in (3, 4, 5, 6)])
    bad = np.arange(len(beams)) % 3 == 0
    if where == "centre":  # a shadow beam's centre does not enter
        bad &= np.arange(len(beams)) % 5 != 4

    def scalars(bs, _):
        bs[bad, abi.B_JP:abi.B_JP + 8] *= 1e3
        col = {"centre": abi.B_CEN + 1, "axis": abi.B_HOR, "direction": abi.B_DIR + 2}.get(where)
        if col is not None:
            bs[bad, col] = value

    def vertex(x, vo):
        if where == "vertex":
            x[vo[:-1][bad] + 1] = value

    spoilt = _batch(abi, beams, src, beam_scalars=scalars, vx=vertex)
    ext = spoilt.beam_external[~bad]
    good = _batch(abi, beams[~bad], src)
    good.beam_external[:] = ext
    grid = abi.Grid.build(np.r_[0.0, np.logspace(-4, -1, 12), np.linspace(0.2, np.pi, 30)], 9)
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        for flags, tol in ((abi.PREC_FP64, 60 * 2.0 ** -53), (abi.INCOHERENT, 60 * 2.0 ** -53),
                           (abi.PREC_MIXED, 60 * 2.0 ** -24),
                           (abi.PREC_MIXED | abi.NO_MFMA, 60 * 2.0 ** -24)):
            ctx.upload(good, consts)
            want = ctx.mueller(flags)[0]
            ctx.upload(spoilt, consts)
            m = ctx.mueller(flags)[0]
            assert np.isfinite(m).all()
            assert np.linalg.norm(m - want) <= tol * np.linalg.norm(want)
