"""The context's shared host copies (csrc/copy_team.h): every byte of every length
arrives, whatever the number of threads; and an uploaded batch whose flag bytes
(the only array of single bytes) go up in shared pieces of awkward lengths."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, load_fixture


def test_every_byte_arrives(tmp_path):
    """Lengths around the 512 KiB from which copies are shared, at 1 to 3 bytes and
    others past whole parts of two, three and four threads, and multiples of a
    page."""
    exe = str(tmp_path / "copy_team")
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-Wall", "-I",
                    os.path.join(ROOT, "mbs-fast_amd", "csrc"),
                    os.path.join(ROOT, "tests", "copy_team_harness.cpp"), "-o", exe], check=True)
    least = 1 << 19
    sizes = [1, 4096, least - 1] + [least + d for d in (0, 1, 2, 3, 4, 4095, 4096)]
    for part in (8192, 12288, 16384):
        for k in (64, 86, 137):
            sizes += [part * k + d for d in (1, 2, 3, part - 1) if part * k >= least]
    p = subprocess.run([exe] + [str(n) for n in sizes], stdout=subprocess.PIPE, text=True,
                       timeout=120)
    assert p.returncode == 0, p.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [1, 2, 3])
def test_flags_of_a_large_batch(pkg, extra):
    """139,250 beams in 16 orientations with 557,056 + extra vertices: the flags'
    piece of a chunk ends 1 to 3 bytes past four equal parts.  Bit for bit against
    page-locked staging, after a batch of the same size whose flags are zero (a
    chunk's former contents); the last edges' flags count in the result."""
    abi = pkg.abi
    fx = load_fixture("sobol_average")
    src, consts = abi.BeamBatch.from_fixture(fx), abi.consts_from_fixture(fx)
    n, want = 139250, 557056 + extra
    four, other = (np.flatnonzero(src.beam_nv == k) for k in (4, 3 if want < 4 * n else 5))
    pick = np.full(n, four[0])
    pick[:abs(want - 4 * n)] = other[0]
    nv = src.beam_nv[pick]
    verts = np.repeat(src.vert_offsets[pick], nv) + np.arange(want) - np.repeat(np.cumsum(nv) - nv,
                                                                               nv)
    beams = dict(orient_offsets=np.r_[np.arange(16) * 8000, n], weights=np.full(16, 1.0 / 16),
                 beam_scalars=src.beam_scalars[pick], beam_nv=nv,
                 beam_external=np.zeros(n, np.int32), vert_offsets=np.r_[0, np.cumsum(nv)],
                 vx=src.vx[verts], vy=src.vy[verts], slope_yx=src.slope_yx[verts],
                 slope_xy=src.slope_xy[verts])
    flags = src.edge_flags[verts]
    batch = abi.BeamBatch(edge_flags=flags, **beams)
    assert int(batch.vert_offsets[-1]) == want
    grid = abi.Grid.build(np.linspace(0.1, 3.0, 5), 4)
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload_staged(batch, consts)
        m = ctx.mueller(abi.PREC_FP64)[0]
        cut = flags.copy()
        cut[-extra:] = 0
        ctx.upload_staged(abi.BeamBatch(edge_flags=cut, **beams), consts)
        assert not np.array_equal(m, ctx.mueller(abi.PREC_FP64)[0])
        ctx.upload(abi.BeamBatch(edge_flags=np.zeros_like(flags), **beams), consts)
        ctx.upload(batch, consts)
        np.testing.assert_array_equal(m, ctx.mueller(abi.PREC_FP64)[0])
