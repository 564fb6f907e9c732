"""Device memory of a batch: what the handler reckons with is what an upload takes,
and a batch that leaves no room for the MFMA operand runs without it."""
import ctypes as C

import numpy as np
import pytest

from conftest import load_fixture


def _copies(abi, n_beams, vertices, n_orient=16):
    """n_beams traced beams of the given vertex count, over and over."""
    fx = load_fixture("config3_aggregate")
    src = abi.BeamBatch.from_fixture(fx)
    pick = np.resize(np.flatnonzero(src.beam_nv == vertices), n_beams)
    verts = (src.vert_offsets[pick][:, None] + np.arange(vertices)).reshape(-1)
    batch = abi.BeamBatch(np.arange(n_orient + 1) * n_beams // n_orient,
                          np.full(n_orient, 1.0 / n_orient), src.beam_scalars[pick],
                          src.beam_nv[pick], src.beam_external[pick],
                          np.arange(n_beams + 1) * vertices, src.vx[verts], src.vy[verts],
                          src.slope_yx[verts], src.slope_xy[verts], src.edge_flags[verts])
    return batch, abi.consts_from_fixture(fx)


@pytest.mark.parametrize("vertices", [3, 4, 5, 7])
def test_batch_size_within_the_budget(pkg, monkeypatch, vertices):
    """The batch size that the handler selects for 0.8 of the free memory is the
    largest power-of-two part of the request that fits in it: input block 304 bytes
    a beam and 33 a vertex, records 1,440 and 64 (csrc/po_layout.h)."""
    abi = pkg.abi
    batch, consts = _copies(abi, 64000, vertices, n_orient=64)
    grid = abi.Grid.build(np.linspace(0.0, np.pi, 5), 4)

    def need(n):
        beams = 1000 * n
        return beams * (304 + 1440) + beams * vertices * (33 + 64) + 64 * grid.cells * 256

    class Lib:
        free = 0

        def mbs_query_memory(self, free, total):
            free._obj.value = total._obj.value = Lib.free
            return 0

    monkeypatch.setattr(pkg.engine, "lib", Lib)
    h = pkg.handler.HandlerPOGpu(grid, consts)
    for n in (64, 32, 8, 2):
        Lib.free = int(need(n) / 0.8) + 2
        assert h.SelectGpuOrientationBatchSize(batch, 0, 64) == n
        Lib.free = int(need(n) / 0.8) - 64
        assert h.SelectGpuOrientationBatchSize(batch, 0, 64) == max(1, n // 2)


@pytest.mark.gpu
@pytest.mark.parametrize("vertices", [4, 7])
def test_bytes_of_an_upload(pkg, vertices):
    """Free memory before and after an upload of 300,000 beams: abi.device_bytes, and
    up to 2 MiB more for each of the seven allocations."""
    abi = pkg.abi
    batch, consts = _copies(abi, 300000, vertices)
    free, total = C.c_int64(), C.c_int64()
    query = pkg.engine.lib().mbs_query_memory
    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(abi.Grid.build(np.linspace(0.0, np.pi, 5), 4))
        assert query(C.byref(free), C.byref(total)) == 0
        before = free.value
        ctx.upload(batch, consts)
        assert query(C.byref(free), C.byref(total)) == 0
    used, said = before - free.value, abi.device_bytes(300000, 300000 * vertices)
    print("%d vertices: %d bytes used, %d said" % (vertices, used, said))
    assert said <= used <= said + 7 * (2 << 20)


@pytest.mark.gpu
def test_batch_without_room_for_the_operand(pkg):
    """4 million beams, 5.5 GB and an operand of 3.1 GB, with the rest of the card
    taken.  With 7.1 GB left the operand finds no room; with all of it there and 1.1
    GB left, the aperture FFT's 1.6 GB take the operand's place.  Both times FP64
    results stay, and the mixed ones are the vector ALU's bit for bit; with memory
    again, the former ones.  What cannot fit in any case (the per-orientation grids
    of 100,000 orientations, 419 GB) is an error and changes nothing."""
    abi = pkg.abi
    batch, consts = _copies(abi, 4000000, 4)
    grid = abi.Grid.build(np.linspace(0.1, 3.0, 7), 12)
    lib, hip = pkg.engine.lib(), C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    taken = []

    def free():
        f, t = C.c_int64(), C.c_int64()
        assert lib.mbs_query_memory(C.byref(f), C.byref(t)) == 0
        return f.value

    def leave(n):  # takes the card's memory but for n bytes
        while free() - n > 2 << 20:
            p = C.c_void_p()
            if hip.hipMalloc(C.byref(p), min(free() - n, 32 << 30)):
                hip.hipGetLastError()
                break
            taken.append(p)
        if not n - (64 << 20) <= free() <= n + (64 << 20):
            pytest.skip("the rest of the card cannot be taken: %d bytes free" % free())

    def give_back():
        while taken:
            hip.hipFree(taken.pop())

    def results(ctx):
        return [ctx.mueller(f)[0] for f in (abi.PREC_FP64, abi.PREC_MIXED,
                                            abi.PREC_MIXED | abi.NO_MFMA)]

    with pkg.engine.Context(0) as ctx:
        ctx.set_grid(grid)
        ctx.upload(batch, consts)
        f64, mfma, valu = results(ctx)
    assert not np.array_equal(mfma, valu)
    with pkg.engine.Context(0) as ctx:
        small, _ = _copies(abi, 1000, 4, n_orient=100000)
        ctx.set_grid(abi.Grid.build(np.linspace(0.0, np.pi, 181), 181))
        ctx.upload(small, consts)
        before = ctx.mueller(abi.PREC_MIXED)[0]
        with pytest.raises(pkg.engine.EngineError, match="memory"):
            ctx.mueller(abi.PREC_FP64 | abi.PER_ORIENT)
        np.testing.assert_array_equal(ctx.mueller(abi.PREC_MIXED)[0], before)
    try:
        with pkg.engine.Context(0) as ctx:
            ctx.set_grid(grid)
            leave(6800 << 20)
            ctx.upload(batch, consts)
            for m, want in zip(results(ctx), (f64, valu, valu)):
                np.testing.assert_array_equal(m, want)
            give_back()
            ctx.upload(batch, consts)
            for m, want in zip(results(ctx), (f64, mfma, valu)):
                np.testing.assert_array_equal(m, want)
            leave(1024 << 20)
            ctx.aperture_fft(np.arange(48), 2048, 4.0, np.zeros((1, 2)), 4)
            for m, want in zip(results(ctx), (f64, valu, valu)):
                np.testing.assert_array_equal(m, want)
    finally:
        give_back()
