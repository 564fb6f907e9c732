"""The work that a user of this engine has it do, as measurable cases.

Every case goes through the package's public entry points (``handler.HandlerPOGpu``
for the calls the reference's host makes once per batch, ``engine.Context`` for
programs that keep a batch resident, ``engine.Mlp`` for the control variate) and
returns what that program gets back: Mueller grids, azimuth-averaged rows, theta
probes, aperture transforms, network outputs and gradients.

Beams come from the reference tracer's own prepared beams (tests/golden/*.npz).
``traced`` batches keep an orientation's beams together: the whole set is turned
about the incident axis by a random angle and scaled, so the shadow beams, the
beams leaving exactly along the poles and the near-singular edges of a traced
particle stay in.  ``resampled`` batches draw beams one by one
(``synthetic.resample``) to the beam counts of large particles.

Mixed-precision results have FP32 accuracy (FP32 phasors and sums) and are kept
as FP32 by the callers here; FP64 results stay FP64.
"""
import math
import os

import numpy as np
import torch

import mbs_loader

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# a (beam, direction) unit's arithmetic without its sincos and reciprocals:
# 169 + 4 nv + 7 nE at nv = nE = 4 (the sets hold 3.9 vertices on average)
UNIT_FLOPS = 213.0
BEAM_BYTES = 36 * 8 + 4 + 4 + 8 + 4 * (4 * 8 + 1)  # host record of a 4-vertex beam
MEAN_BEAMS = {"fixed_absorbing": 185, "config1_fixed": 485, "sobol_average": 231,
              "config5_near_forward": 1468, "config3_aggregate": 4528}
_SOURCES = {}


def _case(name, kind, **kw):
    base = {"kind": kind, "source": "sobol_average", "beams": "traced", "orients": 1,
            "low": 0, "high": 0, "scale": 1.0, "grid": "uniform", "rows": 181, "az": 48,
            "mixed": False, "noshadow": False}
    base.update(kw)
    return dict({"name": name} if name else {}, **base)


def listed():
    return [
        # One orientation of a small absorbing particle on a coarse grid, the
        # smallest call of a fixed-orientation run: launches, copies and waits.
        _case("fixed_absorbing_91x16", "call", source="fixed_absorbing", rows=91, az=16),
        # One orientation of the D = 10 um column on a fine grid, with the
        # no-shadow grid: the reference's fixed-orientation output.
        _case("fixed_column_721x48", "call", source="config1_fixed", rows=721, az=48,
              noshadow=True),
        # One batch of an orientation average from the host's beams to the
        # host's grids, both grids, mixed precision (D = 50 um).
        _case("average_call_mixed", "call", orients=64, scale=5.0, grid="average",
              rows=541, az=96, mixed=True, noshadow=True),
        # The same call in FP64, the default precision of the drop-in.
        _case("average_call_fp64", "call", orients=24, scale=5.0, grid="average", rows=541,
              az=96),
        # The headline workload: 16 orientations of 2,000-15,000 beams each,
        # resident on the device, mixed precision.
        _case("average_large_mixed", "resident", beams="resampled", orients=16, low=2000,
              high=15000, scale=5.0, grid="average", rows=541, az=96, mixed=True),
        # The same particle in FP64, four orientations.
        _case("average_large_fp64", "resident", beams="resampled", orients=4, low=2000,
              high=15000, scale=5.0, grid="average", rows=541, az=96),
        # The 8-column aggregate: 50 to 40,000 beams an orientation, through
        # the device work queue as a replayed graph.
        _case("aggregate_queue_mixed", "queue", source="config3_aggregate", beams="resampled",
              orients=12, low=50, high=40000, grid="average", rows=541, az=96, mixed=True),
        # One size of a multi-size near-forward run (theta 0-5 deg), the beams
        # re-derived on the device.
        _case("size_scan_mixed", "scan", source="config5_near_forward", orients=24, scale=0.35,
              grid="forward", rows=1001, az=48, mixed=True),
        # The theta probe that places a run's zenith grid (incoherent FP64).
        _case("theta_probe", "probe", orients=16, scale=5.0, rows=181, az=48),
        # Per-orientation azimuth-averaged rows, the training data of the
        # control variate and the material of convergence studies.
        _case("training_rows_mixed", "rows", orients=256, rows=181, az=32, mixed=True),
        # The aperture FFT at its largest: 64 beams on 2048 x 2048.
        _case("aperture_fft_2048", "fft", source="config5_near_forward", orients=1, n=2048,
              batch=64, pad=4.0, points=256),
        # The control variate's network: a prediction chunk and a gradient.
        _case("control_variate_net", "net", rows=181, predict=4096, train=512, width=256,
              depth=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "call", "call", "resident", "resident", "resident", "queue",
                       "scan", "probe", "rows", "fft", "net"])
    rows, az = _log(rng, 31, 721), _log(rng, 12, 128)
    scale = round(math.exp(rng.uniform(0.0, math.log(8.0))), 3)
    mixed = rng.random() < 0.6
    if kind == "call":
        fixed = rng.random() < 0.4
        src = rng.choice(["fixed_absorbing", "config1_fixed"]) if fixed else \
            rng.choice(["sobol_average", "sobol_average", "config3_aggregate"])
        return _case(None, kind, source=src, rows=rows, az=az, scale=scale, mixed=mixed,
                     noshadow=rng.random() < 0.4,
                     orients=1 if fixed else _log(rng, 1, 4 if src[:7] == "config3" else 64))
    if kind in ("resident", "queue"):
        agg = kind == "queue" or rng.random() < 0.3
        low = _log(rng, 20, 2000)
        return _case(None, kind, source="config3_aggregate" if agg else "sobol_average",
                     beams="resampled", orients=_log(rng, 1, 12), low=low,
                     high=low + _log(rng, 10, 6000), scale=scale, rows=rows, az=az,
                     grid=rng.choice(["uniform", "average"]),
                     mixed=mixed or kind == "queue", noshadow=rng.random() < 0.25)
    if kind == "scan":
        return _case(None, kind, source="config5_near_forward", orients=_log(rng, 1, 20),
                     scale=round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3), grid="forward",
                     rows=_log(rng, 101, 1001), az=_log(rng, 12, 64), mixed=mixed)
    if kind == "probe":
        return _case(None, kind, orients=_log(rng, 1, 24), scale=scale, rows=_log(rng, 7, 361),
                     az=_log(rng, 12, 96))
    if kind == "rows":
        return _case(None, kind, orients=_log(rng, 8, 300), rows=_log(rng, 46, 361),
                     az=_log(rng, 12, 48), mixed=mixed)
    if kind == "fft":
        return _case(None, kind, source="config5_near_forward", n=1 << rng.randint(7, 11),
                     batch=rng.randint(1, 64), pad=round(rng.uniform(1.5, 8.0), 2),
                     points=_log(rng, 16, 1024))
    return _case(None, kind, rows=_log(rng, 46, 361), predict=_log(rng, 64, 4096),
                 train=_log(rng, 64, 512), width=rng.choice([128, 256]), depth=rng.randint(2, 5))


# ---- inputs -----------------------------------------------------------------

def _source(name):
    if name not in _SOURCES:
        fx = dict(np.load(os.path.join(ROOT, "tests", "golden", name + ".npz")))
        pkg = mbs_loader.load()
        _SOURCES[name] = (pkg.abi.BeamBatch.from_fixture(fx), pkg.abi.consts_from_fixture(fx))
    return _SOURCES[name]


def _theta(case):
    n = case["rows"]
    if case["grid"] == "average":  # dense forward rows, as in the 541-row average grid
        m = max(2, int(round(n * 201.0 / 541.0)))
        return np.radians(np.r_[np.linspace(0.0, 10.0, m),
                                10.0 + 170.0 * np.arange(1, n - m + 1) / (n - m)])
    if case["grid"] == "forward":
        return np.radians(np.linspace(0.0, 5.0, n))
    return np.radians(np.linspace(0.0, 180.0, n))


def _spun(abi, src, picks, angles, scale):
    """Orientations `picks` of src, each turned about the incident axis by its
    angle, with the particle scaled."""
    b = src.subset(list(picks))
    per = np.repeat(np.asarray(angles), np.diff(b.orient_offsets))
    c, s = np.cos(per), np.sin(per)
    bs = b.beam_scalars.copy()
    for col in (abi.B_HOR, abi.B_VER, abi.B_DIR, abi.B_CEN, abi.B_NT, abi.B_NP, abi.B_NXDT,
                abi.B_NXDP, abi.B_NORMAL):
        x, y = bs[:, col].copy(), bs[:, col + 1].copy()
        bs[:, col], bs[:, col + 1] = c * x - s * y, s * x + c * y
    bs[:, abi.B_CEN:abi.B_CEN + 3] *= scale
    bs[:, abi.B_AREA] *= scale * scale
    return abi.BeamBatch(b.orient_offsets, np.full(b.n_orient, 1.0 / b.n_orient), bs, b.beam_nv,
                         b.beam_external, b.vert_offsets, b.vx * scale, b.vy * scale,
                         b.slope_yx, b.slope_xy, b.edge_flags)


def _batch(case, seed):
    """(batch, consts) of a case, from the seed alone."""
    pkg = mbs_loader.load()
    src, consts = _source(case["source"])
    rng = np.random.default_rng(seed)
    n = case["orients"]
    scale = 1.0 if case["kind"] == "scan" else case["scale"]
    if case["beams"] == "traced":
        return _spun(pkg.abi, src, rng.integers(0, src.n_orient, n),
                     rng.uniform(0.0, 2.0 * np.pi, n), scale), consts
    # beam counts: one from each n-th part of the range (uniform for a
    # particle, log-uniform for the aggregate), in a random order
    u = (np.arange(n) + rng.random(n)) / n
    lo, hi = case["low"], case["high"]
    counts = lo * (hi / lo) ** u if case["kind"] == "queue" else lo + (hi - lo) * u
    return pkg.synthetic.resample(src, rng.permutation(counts.astype(np.int64)), scale=scale,
                                  seed=seed), consts


def _net_inputs(case, seed):
    """Parameters (He weights, zero biases), inputs (unit quaternions and log
    size) and standardised targets of the control variate's network."""
    rng = np.random.default_rng(seed)
    dims = [5] + [case["width"]] * case["depth"] + [16 * case["rows"]]
    layers = [(rng.uniform(-1.0, 1.0, (i, o)) * np.sqrt(6.0 / i), np.zeros(o))
              for i, o in zip(dims[:-1], dims[1:])]
    n = case["predict"] + case["train"]
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    q *= np.where(q[:, 3:] < 0, -1.0, 1.0)
    x = np.c_[q, np.log(rng.uniform(10.0, 80.0, n))].astype(np.float32)
    t = rng.normal(size=(case["train"], dims[-1])).astype(np.float32)
    return layers, x[:case["predict"]], x[case["predict"]:], t


def prepare(case, seed):
    pkg = mbs_loader.load()
    abi, kind, s = pkg.abi, case["kind"], {"kind": case["kind"], "mixed": case["mixed"]}
    if kind == "net":
        layers, s["predict"], s["x"], s["t"] = _net_inputs(case, seed)
        s["ctx"] = pkg.engine.Context(0)
        s["net"] = pkg.engine.Mlp(s["ctx"], 5, case["width"], case["depth"], 16 * case["rows"])
        s["net"].set_params(np.concatenate([np.r_[w.ravel(), b] for w, b in layers]))
        return s
    batch, consts = _batch(case, seed)
    s["batch"], s["consts"] = batch, consts
    if kind in ("call", "probe"):
        grid = abi.Grid.build(_theta(case), case["az"])
        s["handler"] = pkg.handler.HandlerPOGpu(grid, consts,
                                                precision="mixed" if case["mixed"] else "fp64")
        s["handler"].SetFullOnly(not case["noshadow"])
        if kind == "probe":
            s["theta"] = _theta(case)
        else:
            shape = (grid.n_az, grid.n_zen + 1, 16)
            s["full"] = np.zeros(shape)
            s["noshadow"] = np.zeros(shape) if case["noshadow"] else None
        return s
    ctx = s["ctx"] = pkg.engine.Context(0)
    s["flags"] = abi.PREC_MIXED if case["mixed"] else abi.PREC_FP64
    if kind == "fft":
        rng = np.random.default_rng([seed, 1])
        s["beams"] = rng.integers(0, batch.n_beams, case["batch"])
        s["ab"] = rng.uniform(-0.1, 0.1, (case["points"], 2)) * np.exp(
            rng.uniform(np.log(1e-2), 0.0, (case["points"], 1)))
        s["n"], s["pad"] = case["n"], case["pad"]
        ctx.upload(batch, consts)
        return s
    ctx.set_grid(abi.Grid.build(_theta(case), case["az"]))
    if kind == "rows":
        s["flags"] |= abi.PER_ORIENT
        return s
    ctx.upload(batch, consts)
    s["want_noshadow"] = case["noshadow"]
    if kind == "queue":
        ctx.set_work_mode(abi.WORK_QUEUE)
        ctx.set_graph(True)
    if kind == "scan":
        nb = batch.n_beams
        ctx.upload_scaling(batch.beam_scalars[:, abi.B_JP:abi.B_JP + 8], np.zeros(nb),
                           np.ones(nb), np.zeros(nb + 1, np.int64), np.zeros(0), 0.0,
                           consts.wave_index)
        s["scale"] = case["scale"]
    return s


def run(state):
    kind = state["kind"]
    if kind == "call":
        # the handler adds into the caller's grids
        full, ns = state["full"], state["noshadow"]
        full[...] = 0.0
        if ns is not None:
            ns[...] = 0.0
        if not state["handler"].HandleOrientationsToLocalGpu(state["batch"], full, ns):
            raise RuntimeError("the batch was refused")
        return _kept(state, full, ns)
    if kind == "probe":
        ok, m11 = state["handler"].DiffractThetasGpu(state["batch"], state["theta"])
        if not ok:
            raise RuntimeError("the batch was refused")
        return m11
    if kind == "net":
        y = state["net"].forward(state["predict"])
        loss, grad = state["net"].gradient(state["x"], state["t"])
        return {"y": y, "loss": np.float32(loss), "grad": grad}
    ctx = state["ctx"]
    if kind == "fft":
        return ctx.aperture_fft(state["beams"], state["n"], state["pad"], state["ab"],
                                4).astype(np.complex64)
    if kind == "rows":
        ctx.upload(state["batch"], state["consts"])
        ctx.diffract(state["flags"])
        return _kept(state, ctx.azimuth_average_per_orient(), None)[0]
    if kind == "scan":
        ctx.rescale(state["scale"])
    return _kept(state, *ctx.mueller(state["flags"], noshadow=state["want_noshadow"]))


def _kept(state, full, noshadow):
    out = [full] if noshadow is None else [full, noshadow]
    return [m.astype(np.float32) for m in out] if state["mixed"] else out


def work(case):
    kind = case["kind"]
    if kind == "net":
        dims = [5] + [case["width"]] * case["depth"] + [16 * case["rows"]]
        mac = sum(i * o for i, o in zip(dims[:-1], dims[1:]))
        n_par = mac + sum(dims[1:])
        rows = case["predict"] + 3 * case["train"]
        return {"bytes": 4.0 * (2 * n_par + (case["predict"] + case["train"]) * (5 + dims[-1])),
                "flops": 2.0 * mac * rows}
    if kind == "fft":
        n = case["n"]
        # the window's rows and columns that can hold a non-zero pixel
        grid = n * n * 8.0
        return {"bytes": case["batch"] * grid * (1.0 + 2.0 / max(1.0, case["pad"])),
                "flops": case["batch"] * 10.0 * n * n * math.log2(n)}
    n = case["orients"]
    if case["beams"] == "traced":
        beams = n * MEAN_BEAMS[case["source"]]
    elif kind == "queue":
        beams = n * (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
    else:
        beams = n * 0.5 * (case["low"] + case["high"])
    cells = case["rows"] * case["az"]
    out = n * case["rows"] * 18 * 8 if kind == "rows" else \
        case["rows"] * 8 if kind == "probe" else cells * 128 * (2 if case["noshadow"] else 1)
    return {"bytes": float(beams * BEAM_BYTES + out), "flops": UNIT_FLOPS * beams * cells}


# ---- the same results in 64 bits, from plain torch ----------------------------

DEVICE = "cuda"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEVICE)


def _directions(theta, n_az, probe):
    """Directions [cells, 3] and rotation vectors u [2, cells, 6], azimuth-major."""
    theta = np.asarray(theta, np.float64)
    phi = np.arange(n_az) * (2.0 * np.pi / n_az)
    st, ct = np.sin(theta)[None, :], np.cos(theta)[None, :]
    d = np.stack([np.cos(phi)[:, None] * st, np.sin(phi)[:, None] * st,
                  np.broadcast_to(-ct, (n_az, len(theta)))], -1)
    vf = np.zeros_like(d)
    vf[..., 0], vf[..., 1] = -np.sin(phi)[:, None], np.cos(phi)[:, None]
    if not probe:
        tol = 256 * np.finfo(np.float64).eps
        vf[:, np.abs(theta - np.pi) <= tol] = (0.0, -1.0, 0.0)
        vf[:, np.abs(theta) <= tol] = (0.0, 1.0, 0.0)
    vt = np.cross(vf, d)
    vt /= np.linalg.norm(vt, axis=-1, keepdims=True)
    u = [np.concatenate([np.cross(v, d), v - d * np.sum(d * v, -1, keepdims=True)], -1)
         for v in (vt, vf)]
    return _t(d.reshape(-1, 3)), _t(np.stack(u).reshape(2, -1, 6))


def _aperture(d, hor, ver, bd, kc, area, px, py, k):
    """Integral of exp(i k (A x + B y)) over each beam's polygon, times
    exp(i psi): complex [beams, cells]; px, py [beams, nv]."""
    A = (bd * hor).sum(1)[:, None] - hor @ d.T
    B = (bd * ver).sum(1)[:, None] - ver @ d.T
    psi = kc @ d.T
    use_b = B.abs() > A.abs()
    inv = 1.0 / (k * torch.where(use_b, B, -A))
    nv = px.shape[1]
    phase = [k * (A * px[:, v, None] + B * py[:, v, None]) for v in range(nv)]
    re, im, big = torch.zeros_like(A), torch.zeros_like(A), torch.zeros_like(A)
    for v in range(nv):
        f = (v + 1) % nv
        step = torch.where(use_b, (px[:, f] - px[:, v])[:, None], (py[:, f] - py[:, v])[:, None])
        mid = 0.5 * (phase[v] + phase[f]) + psi
        amp = step * torch.sinc((phase[f] - phase[v]) * (0.5 / math.pi))
        re -= amp * torch.sin(mid)  # i step sinc e^{i mid}
        im += amp * torch.cos(mid)
        big = torch.maximum(big, phase[v].abs())
    # closed line integrals: of e^{i phi} dx = -i k B I, of e^{i phi} dy = i k A I
    out = torch.complex(re * inv, im * inv)
    small = big <= 1e-3
    if bool(small.any()):  # the moments about the origin, to second order
        x, y = px, py
        xn, yn = torch.roll(x, -1, 1), torch.roll(y, -1, 1)
        cr = x * yn - xn * y
        tw = cr.sum(1)
        safe = torch.where(tw.abs() > 0, tw, torch.ones_like(tw))
        m = lambda w, c: ((w * cr).sum(1) * (2.0 / c) / safe)[:, None]  # noqa: E731
        p1 = k * (A * m(x + xn, 6.0) + B * m(y + yn, 6.0))
        p2 = k * k * (A * A * m(x * x + x * xn + xn * xn, 12.0)
                      + 2.0 * A * B * m(2 * x * y + x * yn + xn * y + 2 * xn * yn, 24.0)
                      + B * B * m(y * y + y * yn + yn * yn, 12.0))
        form = torch.complex(1.0 - 0.5 * p2, p1) * area[:, None] * torch.polar(
            torch.ones_like(psi), psi)
        out = torch.where(small, form, out)
    return out


def _mueller(j):
    """[..., 16] of complex j [..., 2, 2]."""
    a, b, c, e = j[..., 0, 0], j[..., 0, 1], j[..., 1, 0], j[..., 1, 1]
    n = lambda z: z.real ** 2 + z.imag ** 2  # noqa: E731
    r = lambda p, q: (p * q.conj()).real  # noqa: E731
    i = lambda p, q: (p * q.conj()).imag  # noqa: E731
    na, nb, nc, ne = n(a), n(b), n(c), n(e)
    return torch.stack([
        0.5 * (na + nb + nc + ne), 0.5 * (na - nb + nc - ne), -r(a, b) - r(e, c),
        i(e, c) - i(a, b),
        0.5 * (na + nb - nc - ne), 0.5 * (na - nb - nc + ne), r(e, c) - r(a, b),
        -i(a, b) - i(e, c),
        -r(a, c) - r(e, b), r(e, b) - r(a, c), r(a, e) + r(b, c), i(a, e) - i(b, c),
        i(a, c) - i(e, b), i(e, b) + i(a, c), -i(a, e) - i(b, c), r(a, e) - r(b, c)], -1)


def _exact_grids(case, seed, theta, incoherent=False):
    """Per-orientation Mueller grids [n_orient][2][cells, 16] (all beams, all
    but the shadow beams), unweighted, yielded one orientation at a time."""
    batch, consts = _batch(case, seed)
    scale = case["scale"] if case["kind"] == "scan" else 1.0
    bs = batch.beam_scalars.copy()
    bs[:, 9:12] *= scale
    bs[:, 12] *= scale * scale
    k = consts.wave_index
    d, u = _directions(theta, case["az"], incoherent)
    cells = d.shape[0]
    # (i / lambda) with the sign of the area limit
    lead = -(consts.inv_compl_wave[0] + 1j * consts.inv_compl_wave[1])
    if consts.legacy_sign:
        lead = -lead
    ext = batch.beam_external != 0
    g = _t(bs)
    chunk = max(1, int(1.5e7) // cells)
    for o in range(batch.n_orient):
        b0, b1 = int(batch.orient_offsets[o]), int(batch.orient_offsets[o + 1])
        acc = [torch.zeros((cells, 12), dtype=torch.complex128, device=DEVICE) for _ in range(2)]
        inc = torch.zeros((cells, 16), dtype=torch.float64, device=DEVICE)
        ids = np.arange(b0, b1)
        for nv in np.unique(batch.beam_nv[b0:b1]):
            of = ids[batch.beam_nv[b0:b1] == nv]
            for i in range(0, len(of), chunk):
                part = of[i:i + chunk]
                vert = batch.vert_offsets[part][:, None] + np.arange(nv)
                s = g[_t(part)]
                kc = -k * s[:, 9:12] * _t((~ext[part]).astype(np.float64))[:, None]
                f = lead * _aperture(d, s[:, 0:3], s[:, 3:6], s[:, 6:9], kc, s[:, 12],
                                     _t(batch.vx[vert] * scale), _t(batch.vy[vert] * scale), k)
                f = torch.where(torch.isnan(f.real), torch.zeros_like(f), f)
                t = 0.5 * torch.stack([torch.cat([s[:, 13:16], s[:, 19:22]], 1),
                                       torch.cat([s[:, 16:19], s[:, 22:25]], 1)], 1)
                jp = torch.complex(s[:, 25:33:2], s[:, 26:33:2]).reshape(-1, 2, 1, 2)
                w = (t[:, :, :, None] * jp).sum(1)  # [nb, 6, 2]
                if incoherent:
                    for q in range(len(part)):
                        j = torch.einsum("icm,mk->cik", u, w[q].real) + 1j * torch.einsum(
                            "icm,mk->cik", u, w[q].imag)
                        inc += _mueller(j * f[q][:, None, None])
                    continue
                wm = w.reshape(len(part), 12)
                acc[0] += f.T @ wm
                keep = _t((~ext[part]).astype(np.float64))[:, None]
                if case["noshadow"]:
                    acc[1] += f.T @ (wm * keep)
        if incoherent:
            yield [inc]
            continue
        out = []
        for a in acc[:2 if case["noshadow"] else 1]:
            a = a.reshape(cells, 6, 2)
            out.append(_mueller((u[..., None] * a[None]).sum(2).permute(1, 0, 2)))
        yield out


def _exact_rows(grid, theta, n_az):
    """The azimuth average [rows, 18] of a Mueller grid [az, rows, 16]."""
    m = grid.reshape(n_az, len(theta), 4, 4)
    a = -2.0 * torch.arange(n_az, dtype=torch.float64, device=DEVICE) * (2.0 * np.pi / n_az)
    cs, sn = torch.cos(a)[:, None, None], torch.sin(a)[:, None, None]
    r = torch.stack([m[..., 0], m[..., 1] * cs - m[..., 2] * sn, m[..., 1] * sn + m[..., 2] * cs,
                     m[..., 3]], -1)
    tol = 256 * np.finfo(np.float64).eps
    out = r.mean(0).cpu().numpy().reshape(len(theta), 16)
    plain = m.mean(0).cpu().numpy().reshape(len(theta), 16)
    for t, th in enumerate(theta):
        fwd, bwd = abs(th) <= tol, abs(th - np.pi) <= tol
        if fwd or bwd:
            s = plain[t]
            m11 = 0.5 * (s[5] + s[10]) if fwd else 0.5 * (s[5] - s[10])
            o = np.zeros(16)
            o[[0, 5, 10, 15, 3, 12]] = s[0], m11, m11 if fwd else -m11, s[15], s[3], s[3]
            out[t] = o
    edge = np.r_[theta[0], 0.5 * (theta[1:] + theta[:-1]), theta[-1]]
    lo, hi = edge[:-1], edge[1:]
    dcos = 4.0 * np.pi * np.sin(0.5 * (lo + hi)) * np.sin(0.5 * (hi - lo))
    return np.c_[np.degrees(theta), dcos, out]


def _exact_net(case, seed):
    layers, xp, x, t = _net_inputs(case, seed)
    par = []
    for w, b in layers:
        par += [_t(w.astype(np.float32).astype(np.float64)).requires_grad_(), _t(b).requires_grad_()]

    def net(v):
        for i in range(0, len(par), 2):
            v = v @ par[i] + par[i + 1]
            if i + 2 < len(par):
                v = torch.nn.functional.gelu(v)
        return v

    with torch.no_grad():
        y = net(_t(xp.astype(np.float64)))
    loss = ((net(_t(x.astype(np.float64))) - _t(t.astype(np.float64))) ** 2).mean()
    loss.backward()
    return {"y": y.cpu().numpy(), "loss": np.float64(loss.item()),
            "grad": torch.cat([p.grad.reshape(-1) for p in par]).cpu().numpy()}


def _exact_fft(case, seed):
    """The polygons' transforms themselves (the device samples rasters)."""
    batch, consts = _batch(case, seed)
    rng = np.random.default_rng([seed, 1])
    beams = rng.integers(0, batch.n_beams, case["batch"])
    ab = rng.uniform(-0.1, 0.1, (case["points"], 2)) * np.exp(
        rng.uniform(np.log(1e-2), 0.0, (case["points"], 1)))
    # directions d with (b - d).hor = A, (b - d).ver = B for b = 0, hor = x, ver = y
    d = _t(np.c_[-ab, np.zeros(len(ab))])
    e = torch.eye(3, dtype=torch.float64, device=DEVICE)
    z = torch.zeros((1, 3), dtype=torch.float64, device=DEVICE)
    out = []
    for b in beams:
        v = slice(int(batch.vert_offsets[b]), int(batch.vert_offsets[b + 1]))
        area = _t(batch.beam_scalars[b:b + 1, 12])
        out.append(_aperture(d, e[None, 0], e[None, 1], z, z, area, _t(batch.vx[None, v]),
                             _t(batch.vy[None, v]), consts.wave_index)[0])
    return torch.stack(out).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "net":
        return _exact_net(case, seed)
    if kind == "fft":
        return _exact_fft(case, seed)
    theta = _theta(case)
    if kind == "probe":
        th = np.clip(theta, 1e-6, np.pi - 1e-6)
        th = np.where((theta > 1e-14) & (theta < np.pi - 1e-14), theta, th)
        total = sum(g[0] for g in _exact_grids(case, seed, th, incoherent=True))
        m11 = total[:, 0].reshape(case["az"], -1).sum(0)
        return (4.0 * m11 / case["orients"] / (case["az"] + 1)).cpu().numpy()
    if kind == "rows":
        w = 1.0 / case["orients"]
        return np.stack([_exact_rows(g[0] * w, theta, case["az"])
                         for g in _exact_grids(case, seed, theta)])
    total = None
    for g in _exact_grids(case, seed, theta):
        total = g if total is None else [a + b for a, b in zip(total, g)]
    shape = (case["az"], len(theta), 16)
    return [(m / case["orients"]).reshape(shape).cpu().numpy() for m in total]
