// po_math.h -- device math for the PO diffraction kernels (gfx950).
//
// Phasors are evaluated here rather than through the device library so that the
// hot loops' cost and accuracy are known: phases are counted in table nodes, reduced
// against a table in LDS and finished by short polynomials (FP64) or shears
// (FP32, mixed-precision kernels).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mbs {

constexpr double kPi = 3.141592653589793116;            // double(pi) = M_PI
constexpr double kInvTwoPi = 0.15915494309189533577;  // 1 / (2 pi)
// Small-phase switch: every vertex phase within 1e-3 rad
// (HandlerPO_fast.h:161-216).
constexpr double kSmallPhase = 1e-3;
// The mixed-precision kernels' switch.  Their sums cancel to O(phase) of a
// single term where a lane's phase steps are small (kLookStep), so such lanes
// take the moment form where every phase is within 0.25 rad, with polygon moments
// to fifth order (truncation below max|phase|^6 / 6! = 3.4e-7 there).
constexpr double kSmallPhaseMixed = 0.25;

// Slope stored for an edge that is not valid in that direction (|dx| or
// |dy| below the reference's geometric tolerance).  Its coefficient
// A + s B (or s A + B) is then 1e30 times the lane's larger projection, and what
// it adds below 1e-22 of any valid edge's share, so the edge drops out of the sum
// with no per-lane validity test; only a lane with both projections near 1e-30
// (every vertex phase tiny, so it takes the moment form) sees a small coefficient.
constexpr double kInvalidSlope = 1e30;
// One Horner step p*z + c as a single three-operand v_fma_f64 with the
// coefficient in an SGPR pair.  Written as inline assembly because the
// compiler otherwise keeps loop-invariant FP64 coefficients in VGPRs and
// emits v_mov_b64 + v_fmac_f64 (two instructions) for every step.
__device__ __forceinline__ double horner(double p, double z, double c)
{
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(z), "s"(c));
    return r;
}

// ---------------------------------------------------------------------------
// FP64 phasors.  Phases are in nodes, 1/1024 of a turn: a phase is j + r with j =
// rint(p) and |r| <= 1/2.  e^{2 pi i j / 1024} comes from a table in LDS, e^{i d},
// d = 2 pi r / 1024 <= pi / 1024, from Taylor polynomials in r (sin to d^5, cos to
// d^4: the next terms are 5e-22 and 1.2e-18), and one complex product joins them.
// The reduction is three exact additions.  Phases in radians against a 256-entry
// table took one constant more there and a step more in each polynomial; phases
// in turns two moves more, for a product with 1024 whose addend is a constant too.
// ---------------------------------------------------------------------------
constexpr int kTabN = 1024;
// 1.5 2^52: a sum with it carries the integer nearest in its low 32 bits
constexpr double kRoundMagic = 6755399441055744.0;
__device__ __forceinline__ uint32_t low_bits(double t)
{
    return (uint32_t)__builtin_bit_cast(uint64_t, t);
}

// In two halves, so that callers can issue the table reads of several arguments
// before using any of them: reduction and table read, then polynomials and
// product.
__device__ __forceinline__ void node_reduce(double p, const double2 *__restrict__ tab, double &r,
                                            double2 &e)
{
    const double t = p + kRoundMagic;
    r = p - (t - kRoundMagic);
    e = tab[low_bits(t) & (kTabN - 1)];
}

__device__ __forceinline__ void node_poly(double r, double &sd, double &cd)
{
    constexpr double c1 = 6.28318530717958647693 / kTabN, c2 = c1 * c1;
    const double z = r * r;
    const double ps = __builtin_fma(z, c1 * c2 * c2 / 120.0, -c1 * c2 / 6.0);
    sd = r * horner(ps, z, c1);
    const double pc = __builtin_fma(z, c2 * c2 / 24.0, -0.5 * c2);
    cd = __builtin_fma(pc, z, 1.0);
}

__device__ __forceinline__ void node_finish(double r, double2 e, double &s, double &c)
{
    double sd, cd;
    node_poly(r, sd, cd);
    s = __builtin_fma(e.y, cd, e.x * sd);
    c = __builtin_fma(e.x, cd, -(e.y * sd));
}

// The sine alone.
__device__ __forceinline__ double node_sine(double r, double2 e)
{
    double sd, cd;
    node_poly(r, sd, cd);
    return __builtin_fma(e.y, cd, e.x * sd);
}

// ---------------------------------------------------------------------------
// FP32 phasors of the mixed kernels.  A phase is held in nodes (1/1024 turn) as
// an FP64 number with 1.5 2^32 added (kNodeMagic, carried by the phase's constant
// term, so the addition costs nothing): the low word of the sum is then the
// phase modulo 4 turns in units of 2^-30 turn (5.9e-9 rad), exact to that unit
// for phases within 2^21 turns.  Bits 20..29 select one of 1024 nodes, the 20
// bits below are the place between nodes.
//
// Node j lies near (j + 1/2) / 1024 turn, at an angle whose cosine and
// sine / sqrt(2) both happen to be FP32 numbers to ~1/50 ulp (phasor_node_kernel
// looks for it), so that the table adds no rounding; its third word is
// the offset that belongs to that angle.
//
// The rotation by the distance d from the node is three shears, x1 = c - t s,
// s' = s + 2t x1, c' = x1 - t s' with t = d / 2, which is (1 - d^2/2, d) to
// d^3/6 < 5e-9.  With the sine scaled by 1/sqrt(2), in the table and in the
// result, all three take the same factor g = d / sqrt(2): one FMA for g and
// three for the phasor.  (Sine results keep the 1/sqrt(2); the consumers'
// constants absorb the sqrt(2).)  Per vertex this is six vector instructions
// after the phase, where a 512-entry table of (cos, sin, cos/2, sin/2) with an
// FP64 reduction to radians took ten.
// ---------------------------------------------------------------------------
constexpr int kPhasorN = 1024;
constexpr double kNodeMagic = 6442450944.0;              // 1.5 * 2^32
constexpr float kSqrt2 = 1.41421356237309504880f;
constexpr float kInvSqrt2 = 0.70710678118654752440f;
// g = sqrt(2) pi (r - 2^19) 2^-30 - (node offset) / sqrt(2) for the 20-bit place
// r, whose bits taken as an FP32 number are r 2^-149
constexpr double kPhasorHalf = 4.44288293815836624702 / 2048.0;  // at r = 2^19
constexpr float kPhasorG1 = (float)(4.44288293815836624702 * 0x1p+119);
struct __align__(16) PhasorNode {
    float c, s, g0, unused;
};

// The table entry of phase word u (byte offset of a 16-byte entry: bits
// 20..29 of u moved to 4..13, one instruction).
__device__ __forceinline__ PhasorNode phasor_read(uint32_t u, const PhasorNode *__restrict__ tab)
{
    const uint32_t off = (u >> 16) & (uint32_t)((kPhasorN - 1) * sizeof(PhasorNode));
    return *reinterpret_cast<const PhasorNode *>(reinterpret_cast<const char *>(tab) + off);
}

__device__ __forceinline__ float phasor_angle(uint32_t u, PhasorNode e)
{
    // keeps the read at 16 bytes: one of 12 takes 1.6 times the LDS cycles (19.7
    // against 12.0 a wave at random nodes)
    asm volatile("" ::"v"(e.unused));
    return __builtin_fmaf(__uint_as_float(u & 0xfffffu), kPhasorG1, e.g0);
}

// (cos, sin / sqrt 2) of phase word u from its table entry.
__device__ __forceinline__ void phasor_finish(uint32_t u, PhasorNode e, float &c, float &s)
{
    const float g = phasor_angle(u, e);
    const float x1 = __builtin_fmaf(-g, e.s, e.c);
    s = __builtin_fmaf(g, x1, e.s);
    c = __builtin_fmaf(-g, s, x1);
}

// sin / sqrt 2 alone.
__device__ __forceinline__ float sine_finish(uint32_t u, PhasorNode e)
{
    const float g = phasor_angle(u, e);
    return __builtin_fmaf(g, __builtin_fmaf(-g, e.s, e.c), e.s);
}

// Phase steps (in nodes) up to which a lane is looked at one by one for the
// moment form: 0.25 rad, by edge 0's step and then the other edges' half steps.
constexpr double kLookStep = 0.25 * kPhasorN * kInvTwoPi;
// Half steps (in nodes) up to which sin(h) / h is taken from its series; the
// table's relative error grows like 3e-7 / h below.
constexpr float kSeriesStep = 2.0f;

// The phasor of an angle in radians, of any size: reduced to half a turn
// first.
__device__ __forceinline__ void phasor_rad(double x, const PhasorNode *__restrict__ tab,
                                           float &c, float &s)
{
    const double y = x * kInvTwoPi;
    const uint32_t u = low_bits(__builtin_fma(y - __builtin_rint(y), (double)kPhasorN, kNodeMagic));
    phasor_finish(u, phasor_read(u, tab), c, s);
}

// 1/x to full FP64 precision: hardware estimate + two Newton steps.
__device__ __forceinline__ double rcp_f64(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return r;
}

// 1/x from the hardware estimate and one Newton step: relative error below
// (estimate error)^2, about 1e-14 -- used for the edge coefficients, whose
// quotients carry the rounding of ~1e2 rad phase arguments anyway.
__device__ __forceinline__ double rcp_f64_fast(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}

// sin(x)/x from its Taylor series through x^10; for |x| <= 0.25 the first
// omitted term, x^12/13!, is below 4e-18.
__device__ __forceinline__ double sinc_series(double x)
{
    const double z = x * x;
    double p = __builtin_fma(z, -1.0 / 39916800.0, 1.0 / 362880.0);
    p = __builtin_fma(z, p, -1.0 / 5040.0);
    p = __builtin_fma(z, p, 1.0 / 120.0);
    p = __builtin_fma(z, p, -1.0 / 6.0);
    return __builtin_fma(z, p, 1.0);
}

// |k c delta| up to which stable_edge_quotient reads the first phasor alone.
constexpr double kHalfAngle = 0.25;

// add_stable_edge_quotient (src/handler/HandlerPO_fast.h:235-264): the exact
// half-angle form of exp(i phaseStart)(exp(i k c delta) - 1)/c for an edge
// coefficient c at or near zero.  Returns the increment (real part in .x,
// imaginary in .y) so the running sums stay in registers; only lanes at a
// near-singular edge execute it.  The reference evaluates sin(x)/x by a
// short series below |x| = 1e-4 and by the library sine above; here the
// series through x^10 covers |x| <= 0.25 (z = k c delta is below ~1e-4 in
// FP64 and ~0.02 in mixed precision for 50 um beams), and beyond it the plain
// quotient of the two vertex phasors (pr, pi) -> (nr, ni), whose relative
// rounding there is below 1e-12, needs no library call.
__device__ __forceinline__ double2 stable_edge_quotient(double pr, double pi, double nr,
                                                        double ni, double delta, double cc,
                                                        double k)
{
    const double z = k * cc * delta;
    if (__builtin_fabs(z) <= kHalfAngle) {
        const double sh = sinc_series(0.5 * z);
        const double lr = -0.5 * k * k * cc * delta * delta * sh * sh;
        const double li = k * delta * sinc_series(z);
        return make_double2(pr * lr - pi * li, pr * li + pi * lr);
    }
    const double r = rcp_f64(cc);
    return make_double2((nr - pr) * r, (ni - pi) * r);
}

// AddMuellerFromJones (src/math/Mueller.hpp:37-87): out += w * Mueller(J),
// J given as 8 reals (00r 00i 01r 01i 10r 10i 11r 11i).
template <typename T>
__device__ __forceinline__ void add_mueller(double *m, const T *j, double w)
{
    const double j00r = j[0], j00i = j[1], j01r = j[2], j01i = j[3];
    const double j10r = j[4], j10i = j[5], j11r = j[6], j11i = j[7];
    const double a11 = j00r * j00r + j00i * j00i, a12 = j01r * j01r + j01i * j01i;
    const double a21 = j10r * j10r + j10i * j10i, a22 = j11r * j11r + j11i * j11i;
    double A1 = a11 + a21, A2 = a12 + a22;
    m[0] += ((A1 + A2) * 0.5) * w;
    m[1] += ((A1 - A2) * 0.5) * w;
    A1 = a11 - a21;
    A2 = a12 - a22;
    m[4] += ((A1 + A2) * 0.5) * w;
    m[5] += ((A1 - A2) * 0.5) * w;
    double c1r = j00r * j01r + j00i * j01i, c1i = j00i * j01r - j00r * j01i;
    double c2r = j11r * j10r + j11i * j10i, c2i = j11i * j10r - j11r * j10i;
    m[2] += (-c1r - c2r) * w;
    m[3] += (c2i - c1i) * w;
    m[6] += (c2r - c1r) * w;
    m[7] += (-c1i - c2i) * w;
    c1r = j00r * j10r + j00i * j10i;
    c1i = j00i * j10r - j00r * j10i;
    c2r = j11r * j01r + j11i * j01i;
    c2i = j11i * j01r - j11r * j01i;
    m[8] += (-c1r - c2r) * w;
    m[9] += (c2r - c1r) * w;
    m[12] += (c1i - c2i) * w;
    m[13] += (c2i + c1i) * w;
    c1r = j00r * j11r + j00i * j11i;
    c1i = j00i * j11r - j00r * j11i;
    c2r = j01r * j10r + j01i * j10i;
    c2i = j01i * j10r - j01r * j10i;
    m[10] += (c1r + c2r) * w;
    m[11] += (c1i - c2i) * w;
    m[14] += (-c1i - c2i) * w;
    m[15] += (c1r - c2r) * w;
}

}  // namespace mbs
