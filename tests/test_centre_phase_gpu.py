"""The phase that a beam's centre adds to every vertex cancels from the Mueller matrix
of a single beam: FP64, slopes of their own (the reference's edge sums), directions
near the beam's own, where edges' phase steps are small and a rounding of the vertex
phases is large beside them."""
import numpy as np
import pytest

from conftest import load_fixture
from test_pack_gpu import polygon_batch

pytestmark = pytest.mark.gpu


def _bound(abi, b, i, d, k):
    """How far F of beam i may be off, relative to |F|, in directions d.

    A vertex phase within pi, 512 of 1024 nodes, plus a centre phase within 512: two
    fused operations round it by at most half an ulp of 512..1024 nodes each, 2^-43
    nodes = 7.0e-16 rad; table and polynomial leave a phasor 3e-16 more.  So 1e-15 a
    phasor, 2e-15 an edge, over its phase step D: w / D of F = sum w (e^{i phi'} -
    e^{i phi}) / D."""
    s, v = b.beam_scalars[i], slice(b.vert_offsets[i], b.vert_offsets[i + 1])
    x, y = b.vx[v], b.vy[v]
    a_ = (s[abi.B_DIR:abi.B_DIR + 3] - d) @ s[abi.B_HOR:abi.B_HOR + 3]
    b_ = (s[abi.B_DIR:abi.B_DIR + 3] - d) @ s[abi.B_VER:abi.B_VER + 3]
    phi = k * (a_[..., None] * x + b_[..., None] * y)
    step = np.roll(phi, -1, -1) - phi
    use = np.abs(b_) > np.abs(a_)
    w = np.where(use[..., None], np.roll(x, -1) - x, np.roll(y, -1) - y)
    mid = phi + 0.5 * step
    f = (w * np.sinc(step / (2 * np.pi)) * np.exp(1j * mid)).sum(-1)
    with np.errstate(divide="ignore", invalid="ignore"):
        bound = (np.abs(w) * 2e-15 / np.abs(step)).sum(-1) / np.abs(f)
    usable = (np.abs(phi).max(-1) < np.pi) & (np.abs(phi).max(-1) > 1.1e-3) & \
        (np.abs(step).min(-1) > 1e-6)
    return np.where(usable, bound, np.inf)


def test_centre_phase_cancels(pkg):
    abi = pkg.abi
    consts = abi.consts_from_fixture(load_fixture("sobol_average"))
    src = polygon_batch(abi, 58, seed=4)
    n = src.n_beams
    theta = np.logspace(-5, -1, 41)
    grid = abi.Grid.build(theta, 8)
    rng = np.random.default_rng(2)
    result = []
    for centre in (np.zeros((n, 3)), rng.uniform(-60.0, 60.0, (n, 3))):
        bs = src.beam_scalars.copy()
        bs[:, abi.B_CEN:abi.B_CEN + 3] = centre
        batch = abi.BeamBatch(np.arange(n + 1), np.ones(n), bs, src.beam_nv,
                              np.zeros(n, np.int32), src.vert_offsets, src.vx, src.vy,
                              src.slope_yx * (1 + 1e-8), src.slope_xy * (1 + 1e-8),
                              src.edge_flags)
        with pkg.engine.Context(0) as ctx:
            ctx.set_grid(grid)
            ctx.upload(batch, consts)
            ctx.diffract(abi.PREC_FP64 | abi.PER_ORIENT)
            result.append(ctx.per_orient())
    az = np.arange(8) * (2 * np.pi / 8)
    d = np.stack([np.cos(az)[:, None] * np.sin(theta), np.sin(az)[:, None] * np.sin(theta),
                  np.broadcast_to(-np.cos(theta), (8, theta.size))], -1)
    worst, cells = 0.0, 0
    for i in range(n):
        bound = 4.0 * _bound(abi, batch, i, d, consts.wave_index) + 1e-12
        off = np.abs(result[1][i] - result[0][i]).max(-1) / result[0][i][..., 0]
        use = np.isfinite(bound)
        cells += int(use.sum())
        if use.any():
            worst = max(worst, float((off[use] / bound[use]).max()))
    print("%d cells, largest share of the bound %.3f" % (cells, worst))
    assert cells > 1000
    assert worst <= 1.0
