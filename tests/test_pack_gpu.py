"""The device pack and the aperture integral over every vertex count the ABI
takes (3..31), at beam counts around the pack's sixteen beams per workgroup,
against the FP64 oracle.  Half of the beams leave along a pole, so cells near
it take the small-phase moment forms with the packed moments to fifth order.
Bars: those of tests/test_engine_gpu.py for the path (FP64 grid L2 1e-10,
mixed P11 grid L2 1e-4).  No per-cell bar: a single beam's grid has zeros.
"""
import numpy as np
import pytest

import metrics as M
from conftest import load_fixture

pytestmark = pytest.mark.gpu


def polygon_batch(abi, n_beams, seed, scale=1.0):
    """One orientation of n_beams convex polygons with 3, 4, ... 31, 3, ...
    vertices on random ellipses, in the frames and with the polarisation data
    of traced beams; even beams leave along theta = 0."""
    rng = np.random.default_rng(seed)
    src = abi.BeamBatch.from_fixture(load_fixture("sobol_average"))
    bs = src.beam_scalars[rng.integers(0, src.n_beams, n_beams)].copy()
    nv = 3 + np.arange(n_beams) % 29
    vo = np.r_[0, np.cumsum(nv)]
    x, y, syx, sxy, fl = (np.zeros(vo[-1]) for _ in range(5))
    for b in range(n_beams):
        a, c = scale * rng.uniform(0.5, 3.0, 2)
        t = np.sort(rng.uniform(0.0, 2 * np.pi, nv[b]))
        while np.max(np.diff(np.r_[t, t[0] + 2 * np.pi])) > 3.0 or np.min(np.diff(t)) < 1e-3:
            t = np.sort(rng.uniform(0.0, 2 * np.pi, nv[b]))
        v = slice(vo[b], vo[b + 1])
        x[v], y[v] = a * np.cos(t), c * np.sin(t)
        dx, dy = np.roll(x[v], -1) - x[v], np.roll(y[v], -1) - y[v]
        syx[v], sxy[v], fl[v] = dy / dx, dx / dy, 3
        bs[b, abi.B_AREA] = 0.5 * np.sum(x[v] * np.roll(y[v], -1) - np.roll(x[v], -1) * y[v])
        if b % 2 == 0:  # rotate the frame so that the beam leaves along theta = 0
            d = bs[b, abi.B_DIR:abi.B_DIR + 3] / np.linalg.norm(bs[b, abi.B_DIR:abi.B_DIR + 3])
            u = np.array([0.0, 0.0, -1.0]) - d
            n2 = u @ u
            if n2 > 1e-24:  # a reflection is as good as a rotation here
                for col in (abi.B_HOR, abi.B_VER, abi.B_DIR, abi.B_NT, abi.B_NP, abi.B_NXDT,
                            abi.B_NXDP, abi.B_NORMAL):
                    w = bs[b, col:col + 3]
                    bs[b, col:col + 3] = w - 2.0 * u * (u @ w) / n2
    ext = (np.arange(n_beams) % 7 == 6).astype(np.int32)
    return abi.BeamBatch([0, n_beams], [1.0], bs, nv, ext, vo, x, y, syx, sxy, fl)


@pytest.mark.parametrize("n_beams", [1, 15, 16, 17, 31, 64])
def test_every_vertex_count(pkg, oracle, n_beams):
    abi = pkg.abi
    consts = abi.consts_from_fixture(load_fixture("sobol_average"))
    batch = polygon_batch(abi, n_beams, seed=40 + n_beams)
    theta = np.r_[0.0, np.logspace(-6, -1, 21), np.linspace(0.2, np.pi, 40)]
    grid = abi.Grid.build(theta, 7)
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        o, on, _ = oracle.diffract(grid, batch, consts, noshadow=True)
        m, mn = ctx.mueller(abi.PREC_FP64, noshadow=True)
        for a, b in ((m, o), (mn, on)):
            print("%d beams FP64: %s" % (n_beams, M.summary(a, b, theta)))
            assert M.grid_l2(a, b, theta) < 1e-10
        for extra in (0, abi.NO_MFMA):
            m, mn = ctx.mueller(abi.PREC_MIXED | extra, noshadow=True)
            for a, b in ((m, o), (mn, on)):
                e = M.grid_l2(a[..., :1], b[..., :1], theta)
                print("%d beams mixed (%d): P11 grid_l2 %.2e" % (n_beams, extra, e))
                assert e < 1e-4


def _shapes(rng):
    """Polygons of every class of the mixed kernels (and both orientations):
    (name, vertices)."""
    def turn(p, a):
        c, s = np.cos(a), np.sin(a)
        return np.asarray(p) @ np.array([[c, s], [-s, c]])
    out = []
    for _ in range(4):
        a = rng.uniform(0, 2 * np.pi)
        w, h, sk, top = rng.uniform(0.3, 3.0, 4)
        out += [("triangle", turn([(-w, -h), (w, -h), (sk - w, h)], a)),
                ("parallelogram", turn([(-w - sk, -h), (w - sk, -h), (w + sk, h), (sk - w, h)], a)),
                ("trapezoid", turn([(-w, -h), (w, -h), (sk, h), (sk - top, h)], a)),
                ("quadrilateral", turn([(-w, -h), (w, -1.2 * h), (0.9 * w, h), (-w, 0.7 * h)], a)),
                ("rectangle on the axes", np.array([(-w, -h), (w, -h), (w, h), (-w, h)])),
                ("point on an edge", turn([(-w, -h), (0.2 * w, -h), (w, -h), (0.5 * w, h)], a)),
                ("sliver", turn([(-w, -h), (w, -h), (w, 1e-3 - h), (2e-3 - w, 1e-3 - h)], a)),
                ("pentagon", turn([(-w, -h), (w, -h), (1.3 * w, 0), (0, h), (-w, 0.8 * h)], a)),
                ("hexagon", turn([(w * np.cos(t), h * np.sin(t)) for t in np.arange(6) * np.pi / 3],
                                 a))]
    return out


def _class_batch(abi, variant):
    fx = load_fixture("sobol_average")
    consts = abi.consts_from_fixture(fx)
    src = abi.BeamBatch.from_fixture(fx)
    rng, noise = np.random.default_rng(77), np.random.default_rng(78)
    shapes = _shapes(rng)
    bs = src.beam_scalars[rng.integers(0, src.n_beams, len(shapes))].copy()
    cols = {k: [] for k in ("x", "y", "syx", "sxy", "fl")}
    nv = []
    for b, (_, p) in enumerate(shapes):
        p = p * {"tiny": 0.004, "small": 0.1}.get(variant, 1.0)
        if variant == "clockwise":
            p = p[::-1]
        if variant == "doubled":
            p = np.insert(p, 1, p[1], axis=0)
        if variant in ("noise 3e-12", "noise 3e-10"):  # past either tolerance
            size = np.abs(p).max()
            p = p + size * float(variant.split()[1]) * noise.uniform(-1.0, 1.0, p.shape)
        dx, dy = (np.roll(p, -1, 0) - p).T
        okx, oky = np.abs(dx) > 1e-12, np.abs(dy) > 1e-12
        syx = np.divide(dy, dx, out=np.zeros_like(dx), where=okx)
        sxy = np.divide(dx, dy, out=np.zeros_like(dx), where=oky)
        if variant == "slopes":
            syx, sxy = syx * (1 + 1e-4), sxy * (1 + 1e-4)
        for k, v in zip(("x", "y", "syx", "sxy", "fl"),
                        (p[:, 0], p[:, 1], syx, sxy, okx + 2 * oky)):
            cols[k].append(v)
        nv.append(len(p))
        bs[b, abi.B_AREA] = 0.5 * np.sum(p[:, 0] * np.roll(p[:, 1], -1)
                                         - np.roll(p[:, 0], -1) * p[:, 1])
        if b % 3 == 0:  # leaves along theta = 0 (reflect the frame)
            u = np.array([0.0, 0.0, -1.0]) - bs[b, abi.B_DIR:abi.B_DIR + 3]
            for col in (abi.B_HOR, abi.B_VER, abi.B_DIR, abi.B_NT, abi.B_NP, abi.B_NXDT,
                        abi.B_NXDP, abi.B_NORMAL):
                w = bs[b, col:col + 3]
                bs[b, col:col + 3] = w - 2.0 * u * (u @ w) / max(u @ u, 1e-30)
    if variant == "far":
        bs[:, abi.B_CEN:abi.B_CEN + 3] *= 3e5 / np.linalg.norm(bs[:, abi.B_CEN:abi.B_CEN + 3],
                                                               axis=1, keepdims=True)
    if variant == "long axes":
        bs[:, abi.B_HOR:abi.B_HOR + 3] *= 1.5
    nb = len(shapes)
    return consts, abi.BeamBatch([0, nb], [1.0], bs, nv, np.arange(nb) % 5 == 4,
                                 np.r_[0, np.cumsum(nv)],
                                 *[np.concatenate(cols[k]) for k in ("x", "y", "syx", "sxy", "fl")])


@pytest.mark.parametrize("variant", ["plain", "clockwise", "tiny", "small", "far", "slopes",
                                     "doubled", "long axes"])
def test_polygon_classes(pkg, oracle, variant):
    """Shapes of every class on a grid with near-forward rows, as they are; with
    the vertices reversed; scaled to where every direction (tiny) or some
    (small) take the moments; with centres so far out that the phases leave
    the fixed-point range; with slopes that differ from the vertices' by 1e-4;
    with a repeated vertex; with an aperture axis longer than 1."""
    abi = pkg.abi
    consts, batch = _class_batch(abi, variant)
    theta = np.r_[0.0, np.logspace(-4, -1, 25), np.linspace(0.2, np.pi, 40)]
    grid = abi.Grid.build(theta, 9)
    o, on, _ = oracle.diffract(grid, batch, consts, noshadow=True)
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        for extra in (0, abi.NO_MFMA):
            m, mn = ctx.mueller(abi.PREC_MIXED | extra, noshadow=True)
            for a, b in ((m, o), (mn, on)):
                e = M.grid_l2(a, b, theta)
                e11 = M.grid_l2(a[..., :1], b[..., :1], theta)
                print("%s (%d): grid_l2 %.2e, P11 %.2e" % (variant, extra, e, e11))
                # the path's bar; a far centre's phases of 4e6 rad carry 1e-9
                # rad of their own rounding
                assert e11 < 1e-4 and e < 1e-4


@pytest.mark.parametrize("variant", ["plain", "clockwise", "tiny", "small", "far", "slopes",
                                     "doubled", "long axes", "noise 3e-12", "noise 3e-10"])
def test_polygon_classes_fp64(pkg, oracle, variant):
    """The same shapes in FP64, and with vertices moved by 3e-12 and 3e-10 of
    their size, which takes polygons out of one tolerance on parallel edges or
    of both.  eps1 = 0 leaves a lane to the half-angle form only at an edge
    coefficient of zero.  The bar is the path's, but for what the two sides'
    own rounding allows: of phases of 4e6 rad (far), 4e6 2^-53 a step; of the
    sum of O(1) terms that cancel to a phase of 1e-3 squared (tiny), 1e-16 / 1e-6."""
    abi = pkg.abi
    consts, batch = _class_batch(abi, variant)
    bar = {"far": 1e-8, "tiny": 1e-9}.get(variant, 1e-10)
    theta = np.r_[0.0, np.logspace(-4, -1, 25), np.linspace(0.2, np.pi, 40)]
    grid = abi.Grid.build(theta, 9)
    for eps1 in (consts.eps1, 0.0):
        consts.eps1 = eps1
        o, on, _ = oracle.diffract(grid, batch, consts, noshadow=True)
        inc = oracle.incoherent(grid, batch, consts)
        with pkg.engine.Context(0) as ctx:
            ctx.set_grid(grid)
            ctx.upload(batch, consts)
            m, mn = ctx.mueller(abi.PREC_FP64, noshadow=True)
            mi = ctx.mueller(abi.PREC_FP64 | abi.INCOHERENT)
            mi = mi[0] if isinstance(mi, tuple) else mi
        for a, b in ((m, o), (mn, on), (mi, inc)):
            e = M.grid_l2(a, b, theta)
            print("%s, eps1 %g: grid_l2 %.2e" % (variant, eps1, e))
            assert e < bar


@pytest.mark.parametrize("counts", [[1], [3, 1, 700], [0, 5, 0, 64, 1], [40] * 33,
                                    [1] * 30 + [900] + [2] * 40])
@pytest.mark.parametrize("cells", [(3, 1), (13, 5), (120, 300)])
def test_segment_sums(pkg, counts, cells):
    """The sum over beam segments, cut finely and coarsely, against whole
    orientations: orientations of none, one, a few and many segments (fewer
    segments than slices, an orientation across several slices, several in one),
    grids off the multiples of 32 cells and on either side of the mapping's
    tile count.  The same terms in another order: FP64 sums of up to 900 terms
    differ by 900 2^-53 of the largest, mixed ones by 900 2^-24."""
    abi = pkg.abi
    fx = load_fixture("sobol_average")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    batch = pkg.synthetic.resample(src, np.asarray(counts), seed=len(counts))
    theta = np.linspace(0.0, np.pi, cells[0])
    grid = abi.Grid.build(theta, cells[1])
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        for flags, tol in ((abi.PREC_FP64, 1e-12), (abi.PREC_MIXED, 1e-4)):
            ctx.set_work_mode(abi.WORK_ORIENTATIONS)
            want, want_ns = ctx.mueller(flags, noshadow=True)
            for mode in (abi.WORK_SEGMENTS, abi.WORK_QUEUE):
                for target in (1, 500, 65536):
                    ctx.set_work_mode(mode)
                    ctx.set_target_blocks(target)
                    m, mn = ctx.mueller(flags, noshadow=True)
                    for a, b in ((m, want), (mn, want_ns)):
                        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
            ctx.set_work_mode(abi.WORK_SEGMENTS)
            ctx.diffract(flags | abi.PER_ORIENT)
            per = ctx.per_orient()
            full = ctx.mueller(flags)[0]
            assert np.linalg.norm(per.sum(0) - full) <= tol * np.linalg.norm(full)


@pytest.mark.parametrize("shadow", [[], [0], [63, 64], [129], list(range(130))],
                         ids=["none", "first", "edge", "last", "all"])
def test_shadow_beams_apart(pkg, shadow):
    """Shadow beams are looked for 64 at a time and summed apart: at the edges of
    these groups, among 130 beams and in every one of them, the mixed sums
    against the FP64 ones, and the no-shadow grid, which holds none of them.
    Sums of up to 130 FP32 terms, each off by some 2^-22: within 130 2^-22."""
    abi = pkg.abi
    fx = load_fixture("sobol_average")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    batch = pkg.synthetic.resample(src, np.asarray([130, 3]), seed=7)
    batch.beam_external[:] = 0
    batch.beam_external[shadow] = 1
    grid = abi.Grid.build(np.linspace(0.0, np.pi, 37), 6)
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        want, want_ns = ctx.mueller(abi.PREC_FP64, noshadow=True)
        for mode in (abi.WORK_ORIENTATIONS, abi.WORK_SEGMENTS, abi.WORK_QUEUE):
            ctx.set_work_mode(mode)
            m, mn = ctx.mueller(abi.PREC_MIXED, noshadow=True)
            one = ctx.mueller(abi.PREC_MIXED)[0]
            for a, b in ((m, want), (mn, want_ns), (one, want)):
                assert np.linalg.norm(a - b) <= 130 * 2.0 ** -22 * np.linalg.norm(b)
