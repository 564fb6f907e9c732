// po_layout.h -- device-side layout of packed beams and grid tables.
#pragma once

#include <stdint.h>

namespace mbs {

// Beam header, FP64, HDR_STRIDE doubles per beam, wave-uniform reads.  The
// common path of the diffraction kernels reads the beam's EB record instead;
// this serves the lanes and beams that leave it, and the spectrum source.
enum {
    H_HOR = 0,   // aperture horizontal axis (3)
    H_A0 = 3,    // beamDir . hor
    H_VER = 4,   // aperture vertical axis (3)
    H_B0 = 7,    // beamDir . ver
    H_KC = 8,    // -k * centre (3), zero for external beams
    H_PHB = 11,  // max(|A|,|B|) above which some vertex phase exceeds 1e-3 rad
    H_AL = 12,   // small-phase area limit / complWave (complex)
    H_MOM = 14,  // k mX, k mY, k^2 mXX, 2 k^2 mXY, k^2 mYY (5)
    // moments of orders 3, 4, 5 for the mixed kernels' moment form: entry a
    // of order n multiplies A^a B^(n-a) and holds k^n C(n,a) <x^a y^(n-a)> / n!
    H_MOM3 = 19,  // (4)
    H_MOM4 = 23,  // (5)
    H_MOM5 = 28,  // (6)
    H_INV = 34,   // 1 / (F / F') of the mixed class (see EB_SCALE)
    HDR_USED = 35,
    HDR_STRIDE = 36
};

// Polarisation data of a beam, FP64: W[m][c] = s (T0[m] Jp[0][c] + T1[m]
// Jp[1][c]), entry 4m + 2c + r for rotation component m (0..5), Jones column c
// and r = 0 (real part) / 1 (imaginary part); T0 = 1/2 (NT, nxDT), T1 = 1/2 (NP,
// nxDP), Jp = complWave J_phased, s the record's EB_S64.
enum { W64_STRIDE = 24 };

// MFMA B operand of one beam (mixed kernel): the complex contraction
//   G[dir][n] += Re F'(dir) * B[0][n] + Im F'(dir) / sqrt(2) * B[1][n],
// columns n as the W entries above (with s the scale F / F' of the mixed class):
// B[0][n] = (Re W, Im W), B[1][n] = sqrt(2) (-Im W, Re W).  Every B value is
// split into three BF16 parts h + m + l (24 significant bits, nearest rounding);
// record entry [row][n] holds four words of two parts each, the first in the low
// half: (h, m) (h, m) (0, h) (0, l), the partners of the words the kernel makes
// of F's own three parts.
enum { WB_COLS = 24, WB_WORDS = 4, WB_STRIDE = 2 * WB_COLS * WB_WORDS };

// Class of a beam (see "polygon classes" in po_kernels.hip); the class word is
// the vertex count plus BEAM_CLASS times it.
//   BEAM_VERTICES     any other polygon
//   BEAM_TRAPEZOID    a triangle, or a quadrilateral with edges 0 and 2 parallel
//   BEAM_PARALLEL     a parallelogram
//   BEAM_MOMENTS      (mixed kernels) a polygon so small that every direction
//                     takes the moments
//   BEAM_SLOPES       the edge sum with the slopes as given: a polygon whose
//                     slopes or flags say something else than its vertices,
//                     with a degenerate edge, or axes longer than 1
//   BEAM_FAR          (mixed kernels) the same where phases leave the fixed-point
//                     range, and where a value is not finite
enum { BEAM_VERTICES, BEAM_TRAPEZOID, BEAM_PARALLEL, BEAM_MOMENTS, BEAM_SLOPES, BEAM_FAR };
enum { BEAM_CLASS = 32, BEAM_NV = 31 };

// Record of the aperture integral, EB_STRIDE doubles per beam.  Phases and steps
// are in nodes, 1024 to the turn.
enum {
    EB_DIR = 0,    // 1024 b, b the beam direction (3)
    EB_PHASE = 3,  // mixed: -k centre . b, reduced to a turn, plus kNodeMagic (and a
                   // quarter turn for BEAM_TRAPEZOID and BEAM_VERTICES)
    EB_LIM = 4,    // mixed, two FP32: |step| of edge 0 below which a lane is looked at
                   // (BEAM_SLOPES: max(|A|, |B|), in nodes), and below which it
                   // counts as singular
    EB_SCALE = 5,  // mixed, two FP32: (F / F') / EB_S64 and 1 / (F / F'), F' what the
                   // class's formula gives
    EB_KIND = 6,   // the mixed class word; the FP64 class times 2, plus 1 for an
                   // external beam
    EB_VOFF = 7,   // the beam's vertex offset (an integer)
    // phase vectors Q (four, 3 each): -k / 2 pi times points of the aperture (from
    // the particle's origin) or differences of them, the phase being Q . 1024 (d - b)
    // plus the offset.  BEAM_TRAPEZOID: the middle of edge 1, half of edge 1, the
    // middle of the last edge, half of it.  BEAM_PARALLEL: the centre, half of edge
    // 0, half of edge 1.  Others (mixed): -hor / 2 pi, -ver / 2 pi and the beam
    // centre.
    EB_Q = 8,
    EB_PHASE64 = 20,  // the offset for the FP64 kernels (a quarter turn more for
                      // BEAM_TRAPEZOID)
    EB_S64 = 21,      // their F / F'
    EB_LOOK64 = 22,   // their limits: where a lane is looked at (|step| of edge 0, half
    EB_SING64 = 23,   // of it, or max(|A|, |B|) by class), and singular steps
    EB_STRIDE = 24
};

// Vertex records, FP64, 32 bytes: k x, k y, slope dy/dx, slope dx/dy (the
// slopes of edge e = vertex e -> vertex e+1), and 32 more: the edge's dx and dy,
// its two FP32 weights in the mixed kernels (see VX_W) and its flags.  The packed
// vertices start where the beam's class wants its edge 0: at the longest edge,
// or at the longer of a trapezoid's parallel ones.
enum { V_KX = 0, V_KY = 1, V_SYX = 2, V_SXY = 3, VTX_STRIDE = 4 };
// VX_W: -(t_0 x t_e) (1024 k / 2 pi)^2 and none for a quadrilateral, k dx (1024 /
// 2 pi)^2 and -k dy (1024 / 2 pi)^2 from five vertices on.
enum { VX_DX = 0, VX_DY = 1, VX_W = 2, VX_FLAG = 3, VX_STRIDE = 4 };
// Per-vertex edge flags (as the C ABI's MBS_EDGE_VALID_X / _Y): the edge
// from this vertex has a usable dx (enters the |B| > |A| sum) / dy.
enum { EDGE_VX = 1, EDGE_VY = 2 };

// Grid tables, SoA [DT_COUNT][cells], cells in the device's theta-major order.
enum { DT_DIR = 0, DT_U0 = 3, DT_U1 = 9, DT_COUNT = 15 };
// FP32 copies of u0, u1 for the mixed kernels, [cells][DT32_COUNT].
enum { DT32_COUNT = 12 };

// A unit of work: orientations [o_begin, o_end) whole (Mueller mode), or the
// beam range [b_begin, b_end) of orientation o_begin (Jones mode).
struct WorkItem {
    int32_t o_begin;
    int32_t o_end;
    int64_t b_begin;
    int64_t b_end;
};

// Header of the device work queue (work mode MBS_WORK_QUEUE), written by
// plan_segments_kernel: the item count, then for each of the 8 XCDs the end of its
// range of units (unit = item * n_tiles + tile), and the next unit to hand out,
// each in a line of its own (atomics on one line are served one after the other).
enum { Q_ITEMS = 0, Q_END = 1, Q_NEXT = 64, Q_LINE = 64, Q_WORDS = Q_NEXT + 8 * Q_LINE };

}  // namespace mbs
