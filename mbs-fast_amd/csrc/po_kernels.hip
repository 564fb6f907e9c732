// po_kernels.hip -- gfx950 kernels of the PO diffraction engine.
//
// Work mapping.  One lane owns one scattering direction (grid cell, in the
// device's theta-major numbering, see abi_cell); a 256-lane workgroup owns 256
// consecutive cells of one "work item".  A work
// item is either a run of whole orientations (Mueller mode: the lane sums the
// Jones matrices of every beam of an orientation in registers, converts to
// Mueller, and accumulates weight*Mueller over the run) or one segment of one
// orientation's beams (Jones mode, used when there are too few orientations
// to fill the chip: the lane writes the partial Jones sum and a second kernel
// adds the segments and converts).  Every beam of an item is the same for all
// lanes, so beam records are read with wave-uniform loads (scalar cache), and
// all arithmetic per (beam, direction) stays in VGPRs.  Results are reduced
// in a fixed order by separate kernels, so output is bit-reproducible.
//
// Per (beam, direction) the lane evaluates, following the reference CPU loop
// src/handler/HandlerPO.cpp:2632-2776:
//   A = (b - d).hor, B = (b - d).ver                       (k-k0 projected)
//   phi_v = A*k*x_v + B*k*y_v  (+ psi = -k d.c for internal beams, folded into
//   the vertex phasors as the reference CUDA path does, GpuDiffraction.cu:
//   1110-1122), F = complWave * sum_e (e^{i phi_e+1} - e^{i phi_e})/C_e / B
//   (|B|>|A|) or ... / (-A), with the small-phase moment form when
//   max|phi_v| <= 1e-3 and the half-angle form when |C_e| <= eps1;
//   r_ij = u_i(d).T_j(beam) (the Jones rotation of HandlerPO_fast.h:580-683
//   rewritten exactly with per-direction vectors u_i), d = F R J_phased.
// The mixed kernels evaluate the same integral from other sums: see "mixed
// precision" below.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "po_math.h"
#include "po_layout.h"

// Occupancy of the vector-ALU kernels, in waves per SIMD.  FP64: at least 4 (128
// VGPRs), which the common path takes about 120 of with its 24 sums; with 3 waves
// and no spills it is slower (9.5 ms against 8.65 for 35,800 beams on 541 x 96
// directions), since it waits on LDS and scalar loads.  Mixed precision: 7 (72
// VGPRs; 6 with the shadow beams' sums, whose LDS lets no more share a CU).  Left
// alone it takes 75 to 87 and runs at 5 or 6: 4,000 beams of six vertices and more
// on those directions 1.75 ms, with 7 waves 1.52.  Where workgroups take whole
// orientations, 6: the launch ends with the longest, alone on its CU or not (30
// orientations of 800 beams on 181 x 48 directions 0.99 ms with 7, 0.95 with 6 or 5;
// 300 of 230 2.35, 2.34 and 2.47).
// Builds may pass -DMBS_MIN_WAVES=N for tuning (FP64).
#ifndef MBS_MIN_WAVES
#define MBS_MIN_WAVES 4
#endif
#define MBS_OCCUPANCY(waves) __attribute__((amdgpu_waves_per_eu(waves, 8)))
// The MFMA kernel is held to WAVES waves per SIMD (default 5: 96 VGPRs); its
// 29 KB of LDS per workgroup lets five workgroups share a CU.  The autotuner
// also tries 4 and 6 for the default beam-segment kernel.
#ifndef MBS_MFMA_WAVES
#define MBS_MFMA_WAVES 5
#endif
#define MBS_MFMA_OCCUPANCY __attribute__((amdgpu_waves_per_eu(WAVES, 8)))

namespace mbs {

// ---------------------------------------------------------------------------
// Direction cells are numbered theta-major on the device (cell = t n_az + p:
// the azimuths of one theta row are consecutive lanes), while the C ABI's
// grids are azimuth-major (p (n_zen + 1) + t).  Every azimuth cell of a pole
// row has the same direction, and a beam leaving along it meets singular edge
// coefficients there in every such cell; theta-major order keeps those cells
// in two waves instead of one wave per azimuth.  abi_cell maps a device cell
// to its place in the grids the kernels hand back.
// ---------------------------------------------------------------------------
__device__ __forceinline__ size_t abi_cell(int cell, int n_az, int cells)
{
    const int t = cell / n_az;
    const int p = cell - t * n_az;
    return (size_t)p * (cells / n_az) + t;
}

// ---------------------------------------------------------------------------
// Grid tables: per cell dir(3), u0(6), u1(6) as SoA [DT_COUNT][cells].
// u0 = (vt x d, vt - d (d.vt)), u1 = (vf x d, vf - d (d.vf)) with
// vt = (vf x d)/|vf x d| (kept unnormalised when |vf x d|^2 <= 1e-30, as
// rotate_jones_inline does).  Then cpT.vt = NT.(vt x d) + nxDT.(vt - d(d.vt))
// for cpT = d x NT + nxDT - d (d.nxDT), and likewise for cpP, vf.
// ---------------------------------------------------------------------------
// Phasor nodes (po_math.h), one wave per node: of the angles within
// kNodeTries / 2 steps of 2e-7 rad around the nominal one, the angle whose
// cosine and sine / sqrt(2) are nearest to FP32 numbers (the least of the
// larger error, the first of equal ones).
constexpr int kNodeTries = 2048;
__global__ void __launch_bounds__(64) phasor_node_kernel(PhasorNode *__restrict__ tab)
{
    const int j = blockIdx.x;
    const double nominal = (j + 0.5) * (2.0 * kPi / kPhasorN);
    double best = 1.0;
    int at = 0;
    for (int i = threadIdx.x; i < kNodeTries; i += 64) {
        double s, c;
        sincos(nominal + (i - kNodeTries / 2) * 2e-7, &s, &c);
        s *= 0.70710678118654752440;
        const double e = fmax(fabs(c - (float)c), fabs(s - (float)s));
        if (e < best) {
            best = e;
            at = i;
        }
    }
    for (int off = 1; off < 64; off <<= 1) {
        const double e = __shfl_xor(best, off, 64);
        const int i = __shfl_xor(at, off, 64);
        if (e < best || (e == best && i < at)) {
            best = e;
            at = i;
        }
    }
    if (threadIdx.x == 0) {
        const double delta = (at - kNodeTries / 2) * 2e-7;
        double s, c;
        sincos(nominal + delta, &s, &c);
        tab[j] = PhasorNode{(float)c, (float)(s * 0.70710678118654752440),
                            (float)(-kPhasorHalf - delta * 0.70710678118654752440), 0.0f};
    }
}

// e^{2 pi i j / 1024}, the table of the FP64 phasors.
__global__ void turn_table_kernel(double2 *__restrict__ turns)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    double s, c;
    sincospi((double)j / (kTabN / 2), &s, &c);
    turns[j] = make_double2(c, s);
}

__global__ void grid_tables_kernel(const double *__restrict__ theta,
                                   const double *__restrict__ vf, int n_az,
                                   int n_zen1, double az_step,
                                   double *__restrict__ tab, float *__restrict__ tab32)
{
    const int cells = n_az * n_zen1;
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= cells)
        return;
    // device cell order is theta-major (see abi_cell); vf is azimuth-major
    const int t = cell / n_az;
    const int p = cell - t * n_az;
    double st, ct, sp, cp;
    sincos(theta[t], &st, &ct);
    sincos(p * az_step, &sp, &cp);
    const double d[3] = {st * cp, st * sp, -ct};
    const double *vfc = vf + 3 * ((size_t)p * n_zen1 + t);
    const double f[3] = {vfc[0], vfc[1], vfc[2]};
    double vt[3] = {f[1] * d[2] - f[2] * d[1], f[2] * d[0] - f[0] * d[2],
                    f[0] * d[1] - f[1] * d[0]};
    const double l2 = vt[0] * vt[0] + vt[1] * vt[1] + vt[2] * vt[2];
    if (l2 > 1e-30) {
        const double inv = 1.0 / sqrt(l2);
        vt[0] *= inv;
        vt[1] *= inv;
        vt[2] *= inv;
    }
    const double dvt = d[0] * vt[0] + d[1] * vt[1] + d[2] * vt[2];
    const double dvf = d[0] * f[0] + d[1] * f[1] + d[2] * f[2];
    double u[DT_COUNT];
    u[DT_DIR + 0] = d[0];
    u[DT_DIR + 1] = d[1];
    u[DT_DIR + 2] = d[2];
    // u0: (vt x d, vt - d (d.vt))
    u[DT_U0 + 0] = vt[1] * d[2] - vt[2] * d[1];
    u[DT_U0 + 1] = vt[2] * d[0] - vt[0] * d[2];
    u[DT_U0 + 2] = vt[0] * d[1] - vt[1] * d[0];
    u[DT_U0 + 3] = vt[0] - d[0] * dvt;
    u[DT_U0 + 4] = vt[1] - d[1] * dvt;
    u[DT_U0 + 5] = vt[2] - d[2] * dvt;
    u[DT_U1 + 0] = f[1] * d[2] - f[2] * d[1];
    u[DT_U1 + 1] = f[2] * d[0] - f[0] * d[2];
    u[DT_U1 + 2] = f[0] * d[1] - f[1] * d[0];
    u[DT_U1 + 3] = f[0] - d[0] * dvf;
    u[DT_U1 + 4] = f[1] - d[1] * dvf;
    u[DT_U1 + 5] = f[2] - d[2] * dvf;
    for (int q = 0; q < DT_COUNT; ++q)
        tab[(size_t)q * cells + cell] = u[q];
    // FP32 u0, u1 for the mixed kernels (half the bytes per work unit), one
    // 48-byte record per cell
    for (int q = 0; q < DT32_COUNT; ++q)
        tab32[(size_t)cell * DT32_COUNT + q] = (float)u[DT_U0 + q];
}

// ---------------------------------------------------------------------------
// Beam packing, from the C-ABI input arrays to the kernel record
// (po_layout.h): eight lanes per beam, sixteen beams per workgroup.  Small-phase
// moments follow small_phase_polygon_factor (src/handler/HandlerPO_fast.h:154-216).
//
// What bounds it is latency for small batches and issue for large ones.  One
// thread per beam, with the moments (orders 3-5 then) from binomial sums of pow()
// (about 1,800 calls for a 4-vertex beam), took 0.73 ms for 185 beams, 1.74 ms
// for 59,000 and 2.57 ms for 137,000; this form takes 13, 53 and 105 us.  The
// polygon is staged in LDS, the lanes of a group
// take the vertices in turn and add their sums by butterflies, and an edge's
// share of a moment is a 3-point Gauss rule: over the triangle (0, P, Q) a
// monomial of degree n integrates to det(P, Q) / (n + 2) times its mean along
// PQ, which three nodes give exactly to degree 5.  The record goes through LDS
// so that its stores are contiguous.
// ---------------------------------------------------------------------------
enum { PACK_GROUP = 8, PACK_BEAMS = 16, PACK_THREADS = PACK_GROUP * PACK_BEAMS };

__device__ __forceinline__ double group_sum(double v)
{
    for (int off = 1; off < PACK_GROUP; off <<= 1)
        v += __shfl_xor(v, off, PACK_GROUP);
    return v;
}

__device__ __forceinline__ double group_min(double v)
{
    for (int off = 1; off < PACK_GROUP; off <<= 1)
        v = fmin(v, __shfl_xor(v, off, PACK_GROUP));
    return v;
}

// FP32 -> BF16 bits, nearest (ties to even), and back.
__device__ __forceinline__ uint32_t bf16_bits(float x)
{
    const uint32_t u = __float_as_uint(x);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_value(uint32_t b) { return __uint_as_float(b << 16); }

// Two 32-bit values in one FP64 slot (low word first).
__device__ __forceinline__ double pack_words(uint32_t lo, uint32_t hi)
{
    return __builtin_bit_cast(double, (uint64_t)lo | (uint64_t)hi << 32);
}
__device__ __forceinline__ double pack_floats(float lo, float hi)
{
    return pack_words(__float_as_uint(lo), __float_as_uint(hi));
}
__device__ __forceinline__ int low_word(double slot)
{
    return (int)(uint32_t)__builtin_bit_cast(uint64_t, slot);
}
__device__ __forceinline__ int high_word(double slot)
{
    return (int)(uint32_t)(__builtin_bit_cast(uint64_t, slot) >> 32);
}
__device__ __forceinline__ float low_float(double slot)
{
    return __uint_as_float((uint32_t)__builtin_bit_cast(uint64_t, slot));
}
__device__ __forceinline__ float high_float(double slot)
{
    return __uint_as_float((uint32_t)(__builtin_bit_cast(uint64_t, slot) >> 32));
}

__global__ void __launch_bounds__(PACK_THREADS) pack_beams_kernel(
    int n_beams, const double *__restrict__ bs, const int32_t *__restrict__ nv_in,
    const int32_t *__restrict__ ext_in, const int64_t *__restrict__ voff,
    const double *__restrict__ vx, const double *__restrict__ vy,
    const double *__restrict__ syx, const double *__restrict__ sxy,
    const uint8_t *__restrict__ ef, double k, double al_re, double al_im, double cw_re,
    double cw_im, double sc, const double *__restrict__ raw_j,
    const double *__restrict__ path, const double *__restrict__ sign,
    const int64_t *__restrict__ abs_off, const double *__restrict__ abs_path, double c_abs,
    double k_j, double eps1, double eps_mixed, double *__restrict__ hdr,
    double *__restrict__ w64, double *__restrict__ vtx, double *__restrict__ vx_out,
    uint32_t *__restrict__ wb, double *__restrict__ ebeam)
{
    __shared__ double s_bs[PACK_BEAMS * 36];
    __shared__ double s_x[PACK_BEAMS][33], s_y[PACK_BEAMS][33];  // odd stride: no bank conflicts
    __shared__ double s_h[PACK_BEAMS * HDR_STRIDE];
    __shared__ double s_jp[PACK_BEAMS][8];  // complWave * J_phased
    __shared__ double s_s64[PACK_BEAMS], s_scale[PACK_BEAMS];
    const int g = threadIdx.x / PACK_GROUP, q = threadIdx.x % PACK_GROUP;
    const int first = blockIdx.x * PACK_BEAMS;
    const int count = min((int)PACK_BEAMS, n_beams - first);  // beams of this workgroup
    const int b = first + min(g, count - 1);  // spare groups repeat the last beam
    for (int i = threadIdx.x; i < count * 36; i += PACK_THREADS)
        s_bs[i] = bs[(size_t)first * 36 + i];
    const int nv = nv_in[b];
    const int64_t v0 = voff[b];
    // size rescaling (raw_j set): vertices and centre times sc, area times
    // sc^2, J_phased rebuilt below; sc = 1 leaves every value as it is
    for (int i = q; i < nv; i += PACK_GROUP) {
        s_x[g][i] = vx[v0 + i] * sc;
        s_y[g][i] = vy[v0 + i] * sc;
    }
    __syncthreads();
    const double *s = s_bs + (b - first) * 36, *px = s_x[g], *py = s_y[g];
    double *h = s_h + g * HDR_STRIDE;
    // polygon sums about the aperture origin, and the bounding box
    double sum[6] = {0, 0, 0, 0, 0, 0}, m3[4] = {0, 0, 0, 0}, m4[5] = {0, 0, 0, 0, 0},
           m5[6] = {0, 0, 0, 0, 0, 0};
    double minX = 1e300, maxX = -1e300, minY = 1e300, maxY = -1e300;
    double longest = -1.0;  // squared length of this lane's longest edge, and
    int start = 0;          // the edge (the least index of equal ones)
    for (int i = q; i < nv; i += PACK_GROUP) {
        const int j = (i + 1 < nv) ? i + 1 : 0;
        const double xi = px[i], yi = py[i], xj = px[j], yj = py[j];
        const double cr = xi * yj - xj * yi;
        sum[0] += cr;
        sum[1] += (xi + xj) * cr;
        sum[2] += (yi + yj) * cr;
        sum[3] += (xi * xi + xi * xj + xj * xj) * cr;
        sum[4] += (yi * yi + yi * yj + yj * yj) * cr;
        sum[5] += (2.0 * xi * yi + xi * yj + xj * yi + 2.0 * xj * yj) * cr;
        minX = fmin(minX, xi);
        maxX = fmax(maxX, xi);
        minY = fmin(minY, yi);
        maxY = fmax(maxY, yi);
        const double l2 = (xj - xi) * (xj - xi) + (yj - yi) * (yj - yi);
        if (l2 > longest) {
            longest = l2;
            start = i;
        }
        const double node[3] = {0.5 - 0.38729833462074168852, 0.5,
                                0.5 + 0.38729833462074168852};
        const double weight[3] = {5.0 / 18.0, 8.0 / 18.0, 5.0 / 18.0};
        for (int n = 0; n < 3; ++n) {
            const double x = xi + node[n] * (xj - xi), y = yi + node[n] * (yj - yi);
            double powx[6], powy[6];  // the weight in those of x
            powx[0] = weight[n] * cr;
            powy[0] = 1.0;
            for (int e = 1; e < 6; ++e) {
                powx[e] = powx[e - 1] * x;
                powy[e] = powy[e - 1] * y;
            }
            for (int e = 0; e < 4; ++e)
                m3[e] += powx[e] * powy[3 - e];
            for (int e = 0; e < 5; ++e)
                m4[e] += powx[e] * powy[4 - e];
            for (int e = 0; e < 6; ++e)
                m5[e] += powx[e] * powy[5 - e];
        }
    }
    for (double &v : sum)
        v = group_sum(v);
    for (double &v : m3)
        v = group_sum(v);
    for (double &v : m4)
        v = group_sum(v);
    for (double &v : m5)
        v = group_sum(v);
    for (int off = 1; off < PACK_GROUP; off <<= 1) {
        const double l2 = __shfl_xor(longest, off, PACK_GROUP);
        const int at = __shfl_xor(start, off, PACK_GROUP);
        if (l2 > longest || (l2 == longest && at < start)) {
            longest = l2;
            start = at;
        }
    }
    minX = group_min(minX);
    minY = group_min(minY);
    maxX = -group_min(-maxX);
    maxY = -group_min(-maxY);
    const double tw = sum[0];
    const double areaScale = fmax((maxX - minX) * (maxY - minY), 2.2250738585072014e-308);
    const double inv = !(fabs(tw) <= 0x1p-40 * areaScale) ? 2.0 / tw : 0.0;
    // Small-phase bound.  The vertex phases k (A x + B y) spread over at
    // least k |(A, B)| w, w the least width of the vertex set, so some phase
    // exceeds 1e-3 rad once max(|A|, |B|) > 2e-3 / (k w); the kernels test
    // the vertices one by one only below that (2 % margin for rounding).  w
    // is the least, over all vertex pairs, of the other vertices' spread
    // across the line through the pair: every edge of the convex hull is such
    // a pair, and the hull's least width lies across one of its edges.
    double wmin = __builtin_inf();
    for (int i = q; i < nv; i += PACK_GROUP) {
        const double xi = px[i], yi = py[i];
        for (int j = i + 1; j < nv; ++j) {
            const double ex = px[j] - xi, ey = py[j] - yi;
            const double len = sqrt(ex * ex + ey * ey);
            if (!(len > 0.0))
                continue;
            double lo = 0.0, hi = 0.0;
            for (int l = 0; l < nv; ++l) {
                const double c = ex * (py[l] - yi) - ey * (px[l] - xi);
                lo = fmin(lo, c);
                hi = fmax(hi, c);
            }
            wmin = fmin(wmin, (hi - lo) / len);
        }
    }
    wmin = group_min(wmin);
    const bool ext = ext_in[b] != 0;
    const double *hor = s + 0, *ver = s + 3, *bd = s + 6;
    if (q == 0) {
        for (int i = 0; i < 3; ++i) {
            h[H_HOR + i] = hor[i];
            h[H_VER + i] = ver[i];
            // psi = -k d.c for internal beams; external beams carry no
            // direction phase
            h[H_KC + i] = ext ? 0.0 : -k * (s[9 + i] * sc);
        }
        h[H_A0] = bd[0] * hor[0] + bd[1] * hor[1] + bd[2] * hor[2];
        h[H_B0] = bd[0] * ver[0] + bd[1] * ver[1] + bd[2] * ver[2];
        // complWave is folded into J_phased below; the small-phase area limit is
        // therefore stored divided by complWave.
        const double area = s[12] * (sc * sc);
        const double cw2 = cw_re * cw_re + cw_im * cw_im;
        const double lr = al_re * area, li = al_im * area;
        h[H_AL + 0] = (lr * cw_re + li * cw_im) / cw2;
        h[H_AL + 1] = (li * cw_re - lr * cw_im) / cw2;
        // a degenerate or very large polygon keeps the per-vertex test everywhere
        const double phb =
            (wmin > 0.0 && wmin < __builtin_inf()) ? 2.04e-3 / (k * wmin) : __builtin_inf();
        h[H_PHB] = phb;
        for (int i = HDR_USED; i < HDR_STRIDE; ++i)
            h[i] = 0.0;
    } else if (q == 1) {
        // entry a of order n: k^n C(n, a) <x^a y^(n-a)> / n!, the mean being
        // the integral over the polygon divided by its area tw / 2
        h[H_MOM + 0] = k * ((sum[1] / 6.0) * inv);
        h[H_MOM + 1] = k * ((sum[2] / 6.0) * inv);
        h[H_MOM + 2] = k * k * ((sum[3] / 12.0) * inv);
        h[H_MOM + 3] = 2.0 * k * k * ((sum[5] / 24.0) * inv);
        h[H_MOM + 4] = k * k * ((sum[4] / 12.0) * inv);
        const double k3 = k * k * k;
        const double c3[4] = {1, 3, 3, 1}, c4[5] = {1, 4, 6, 4, 1}, c5[6] = {1, 5, 10, 10, 5, 1};
        for (int a = 0; a < 4; ++a)
            h[H_MOM3 + a] = k3 * c3[a] * (m3[a] / 5.0 * inv) / 6.0;
        for (int a = 0; a < 5; ++a)
            h[H_MOM4 + a] = k3 * k * c4[a] * (m4[a] / 6.0 * inv) / 24.0;
        for (int a = 0; a < 6; ++a)
            h[H_MOM5 + a] = k3 * k * k * c5[a] * (m5[a] / 7.0 * inv) / 120.0;
    }
    // J_phased, or for a rescaled set sign * a(sc) * J * exp(i k_j path sc),
    // a(sc) the mean of exp(c_abs p sc) over the absorption paths p (1 for
    // p <= DBL_EPSILON): the host rule of the multi-size pack
    double amp = 1.0, sn = 0.0, cs = 1.0;
    if (raw_j) {
        amp = sign[b];
        const int64_t a0 = abs_off[b], a1 = abs_off[b + 1];
        if (a1 > a0) {
            double total = 0.0;
            for (int64_t a = a0 + q; a < a1; a += PACK_GROUP)
                total +=
                    abs_path[a] > 2.220446049250313e-16 ? exp(c_abs * abs_path[a] * sc) : 1.0;
            amp *= group_sum(total) / (double)(a1 - a0);
        }
        sincos(k_j * (path[b] * sc), &sn, &cs);
    }
    if (q < 4) {  // complWave * J_phased, one complex element a lane
        double jr, ji;
        if (raw_j) {
            const double rr = raw_j[(size_t)b * 8 + 2 * q] * amp;
            const double ri = raw_j[(size_t)b * 8 + 2 * q + 1] * amp;
            jr = rr * cs - ri * sn;
            ji = rr * sn + ri * cs;
        } else {
            jr = s[25 + 2 * q];
            ji = s[26 + 2 * q];
        }
        s_jp[g][2 * q] = cw_re * jr - cw_im * ji;
        s_jp[g][2 * q + 1] = cw_re * ji + cw_im * jr;
    }
    // The beam's class.  The formulas work from the vertices alone, so the
    // slopes and flags have to agree with them (an edge left out of one branch of
    // the reference's sum must be negligible in it), and in the mixed kernels the
    // phases have to fit the fixed-point range; any other beam keeps the sum over
    // the slopes.  "Agree" and "parallel" are 1e-9 for the mixed kernels and 1e-13
    // for the FP64 ones, the size of their own rounding for phases of 1e2-1e3 rad.
    // (Of a traced hexagonal column's quadrilaterals 0.945 have a parallel pair
    // to 1e-13 and 0.964 to 1e-12 or any tolerance up to 1e-6.)
    const double lmax = sqrt(longest);
    const double cx = ext ? 0.0 : s[9] * sc, cy = ext ? 0.0 : s[10] * sc,
                 cz = ext ? 0.0 : s[11] * sc;
    const double k_turn = k * kInvTwoPi, k_node = kPhasorN * k_turn;
    const double tol = 1e-9 * lmax;
    // 2 where every edge agrees closely, 1 where every edge does; the largest
    // |vertex|; 1 where every value is finite
    double agree = 2.0, reach = 0.0, finite = 1.0;
    for (int i = 0; i < 9; ++i)
        finite = fabs(s[i]) < __builtin_inf() ? finite : 0.0;
    finite = fabs(k * cx) + fabs(k * cy) + fabs(k * cz) < __builtin_inf() ? finite : 0.0;
    for (int i = q; i < nv; i += PACK_GROUP) {
        const int to = (i + 1 < nv) ? i + 1 : 0;
        const double x = px[i], y = py[i], dx = px[to] - x, dy = py[to] - y;
        const uint8_t f = ef[v0 + i];
        const double offx = fabs((f & 1) ? syx[v0 + i] * dx - dy : dx);
        const double offy = fabs((f & 2) ? sxy[v0 + i] * dy - dx : dy);
        const bool edge = sqrt(dx * dx + dy * dy) > tol && (f & 3);
        const double here = !(edge && offx <= tol && offy <= tol) ? 0.0
                            : offx <= 1e-4 * tol && offy <= 1e-4 * tol ? 2.0 : 1.0;
        agree = fmin(agree, here);
        reach = fmax(reach, sqrt(x * x + y * y));
        finite = fabs(k * x) + fabs(k * y) < __builtin_inf() ? finite : 0.0;
    }
    agree = group_min(agree);
    finite = group_min(finite);
    reach = -group_min(-reach);
    const double n_hor = hor[0] * hor[0] + hor[1] * hor[1] + hor[2] * hor[2];
    const double n_ver = ver[0] * ver[0] + ver[1] * ver[1] + ver[2] * ver[2];
    const double n_bd = bd[0] * bd[0] + bd[1] * bd[1] + bd[2] * bd[2];
    const double skew = hor[0] * ver[0] + hor[1] * ver[1] + hor[2] * ver[2];
    // |phase| <= |Q| |d - b| with axes no longer than 1; comparisons written
    // so that a value that is not a number fails them
    const bool unit = n_hor <= 1.0 + 1e-6 && n_ver <= 1.0 + 1e-6 && n_bd <= 1.0 + 1e-6;
    const double far = sqrt(cx * cx + cy * cy + cz * cz);
    const bool fits = 2.5 * k_turn * (far + reach) < 0x1p20;
    // the same for any axes, |d - b| <= 1 + |b|
    const bool in_range = 1.25 * k_turn * (far + (sqrt(n_hor) + sqrt(n_ver)) * reach) *
                              (1.0 + sqrt(n_bd)) < 0x1p20;
    // the polygon's own form, and edge 0 for it
    int form = BEAM_VERTICES, from = start;
    bool close = agree == 2.0;  // to the FP64 kernels' tolerance
    const auto cross = [&](int i, int j) {
        const int i1 = (i + 1) % nv, j1 = (j + 1) % nv;
        return (px[i1] - px[i]) * (py[j1] - py[j]) - (py[i1] - py[i]) * (px[j1] - px[j]);
    };
    const auto len2 = [&](int i) {
        const int i1 = (i + 1) % nv;
        return (px[i1] - px[i]) * (px[i1] - px[i]) + (py[i1] - py[i]) * (py[i1] - py[i]);
    };
    if (nv == 3) {
        form = BEAM_TRAPEZOID;
    } else if (nv == 4) {
        // parallel edges, against the area's own products
        const double c02 = fabs(cross(0, 2)) / fmin(fabs(cross(0, 1)), fabs(cross(0, 3)));
        const double c13 = fabs(cross(1, 3)) / fmin(fabs(cross(0, 1)), fabs(cross(2, 1)));
        const double gx = px[0] - px[1] + px[2] - px[3], gy = py[0] - py[1] + py[2] - py[3];
        const double gap = k * sqrt(gx * gx + gy * gy);
        const bool para = c02 <= 1e-9 && c13 <= 1e-9 && gap <= 1e-8;
        const bool para64 = para && gap <= 4e-15 * k * (reach + sqrt(cx * cx + cy * cy + cz * cz));
        const double c = fmin(c02, c13);
        if (para && (para64 || !(c <= 1e-13))) {
            form = BEAM_PARALLEL;
            close = close && para64;
        } else if (c <= 1e-9) {
            form = BEAM_TRAPEZOID;
            close = close && c <= 1e-13;
            // the pair that is parallel, the nearer to it of two
            from = c02 <= c13 ? (len2(0) >= len2(2) ? 0 : 2) : (len2(1) >= len2(3) ? 1 : 3);
        }
    }
    double s64 = 1.0, scale = 1.0;  // F / F' of the formulas, FP64 and mixed
    int cls64 = BEAM_SLOPES, cls = BEAM_VERTICES;
    if (form != BEAM_VERTICES) {
        // w_1 = -(t_0 x t_1) (1024 k / 2 pi)^2, steps being in nodes
        const double w1 = -cross(from, (from + 1) % nv) * k_node * k_node;
        if (fabs(w1) >= 1e-30 && fabs(w1) <= 1e30) {
            if (unit && agree >= 1.0)
                start = from;
            if (unit && close && finite == 1.0) {
                cls64 = form;  // else the sum over vertices, below
                s64 = form == BEAM_PARALLEL ? -w1 : w1;
            }
            // the mixed kernels' sines carry 1/sqrt(2) each
            scale = form == BEAM_PARALLEL ? -2.0 * w1 : 1.41421356237309504880 * w1;
            cls = form;
        } else if (nv == 3) {
            cls = BEAM_SLOPES;
        }
    }
    if (cls64 == BEAM_SLOPES && unit && agree == 2.0 && finite == 1.0) {
        cls64 = BEAM_VERTICES;
        s64 = k_node * (kPhasorN * kInvTwoPi);
    }
    if (!(unit && fits && agree >= 1.0) || finite != 1.0)
        cls = in_range && finite == 1.0 && cls64 == BEAM_SLOPES ? BEAM_SLOPES : BEAM_FAR;
    else if (fabs(skew) <= 1e-6 && 2.01 * k * reach <= kSmallPhaseMixed)
        cls = BEAM_MOMENTS;
    if (cls == BEAM_VERTICES)
        scale = 1.41421356237309504880;
    else if (cls >= BEAM_MOMENTS)
        scale = 1.0;
    // phase vector in turns of a point of the aperture plane, from the beam
    // centre or from the particle's origin
    const auto turns = [&](double x, double y, bool centred, double *out) {
        for (int i = 0; i < 3; ++i)
            out[i] = -k_turn * ((centred ? 0.0 : i == 0 ? cx : i == 1 ? cy : cz) + x * hor[i] +
                                y * ver[i]);
    };
    const auto vert = [&](int i) {  // vertex i of the record
        const int at = start + i;
        return at < nv ? at : at - nv;
    };
    const double t0x = px[vert(1)] - px[vert(0)], t0y = py[vert(1)] - py[vert(0)];
    for (int i = q; i < nv && g < count; i += PACK_GROUP) {
        const int at = vert(i), to = (at + 1 < nv) ? at + 1 : 0;
        const double x = px[at], y = py[at], dx = px[to] - x, dy = py[to] - y;
        const uint8_t f = ef[v0 + at];
        double *v = vtx + (size_t)(v0 + i) * VTX_STRIDE;
        v[V_KX] = k * x;
        v[V_KY] = k * y;
        v[V_SYX] = (f & 1) ? syx[v0 + at] : kInvalidSlope;
        v[V_SXY] = (f & 2) ? sxy[v0 + at] : kInvalidSlope;
        double *w = vx_out + (size_t)(v0 + i) * VX_STRIDE;
        w[VX_DX] = dx;
        w[VX_DY] = dy;
        const double tx = t0x * k_node, ty = t0y * k_node;
        const double kw = k_node * (kPhasorN * kInvTwoPi);
        w[VX_W] = nv == 4 ? pack_floats(i == 0 ? 0.0f : (float)((ty * dx - tx * dy) * k_node), 0.0f)
                          : pack_floats((float)(kw * dx), (float)(-kw * dy));
        w[VX_FLAG] = pack_words(f, 0);
    }
    if (q == 0 && g < count) {
        const auto X = [&](int i) { return px[vert(i % nv)]; };
        const auto Y = [&](int i) { return py[vert(i % nv)]; };
        double *eb = ebeam + (size_t)b * EB_STRIDE, *eq = eb + EB_Q;
        const bool trapezoid = cls == BEAM_TRAPEZOID || cls64 == BEAM_TRAPEZOID;
        const bool parallel = cls == BEAM_PARALLEL || cls64 == BEAM_PARALLEL;
        if (trapezoid) {  // edge 1 and the last one
            turns(0.5 * (X(1) + X(2)), 0.5 * (Y(1) + Y(2)), false, eq);
            turns(0.5 * (X(2) - X(1)), 0.5 * (Y(2) - Y(1)), true, eq + 3);
            turns(0.5 * (X(nv - 1) + X(0)), 0.5 * (Y(nv - 1) + Y(0)), false, eq + 6);
            turns(0.5 * (X(0) - X(nv - 1)), 0.5 * (Y(0) - Y(nv - 1)), true, eq + 9);
        } else if (parallel) {
            // means over opposite vertices and edges: what the polygon lacks to a
            // parallelogram then enters in pairs of opposite sign
            const double ux = X(1) - X(0) + (X(2) - X(3)), uy = Y(1) - Y(0) + (Y(2) - Y(3));
            const double wx = X(2) - X(1) + (X(3) - X(0)), wy = Y(2) - Y(1) + (Y(3) - Y(0));
            turns(0.25 * (X(0) + X(2) + (X(1) + X(3))), 0.25 * (Y(0) + Y(2) + (Y(1) + Y(3))), false,
                  eq);
            turns(0.25 * ux, 0.25 * uy, true, eq + 3);
            turns(0.25 * wx, 0.25 * wy, true, eq + 6);
            eq[9] = eq[10] = eq[11] = 0.0;
        } else {
            for (int i = 0; i < 3; ++i) {
                eq[i] = -kInvTwoPi * hor[i];
                eq[3 + i] = -kInvTwoPi * ver[i];
                eq[9 + i] = 0.0;
            }
            turns(0.0, 0.0, false, eq + 6);
        }
        const double offset = -k_turn * (cx * bd[0] + cy * bd[1] + cz * bd[2]);
        const double part = kPhasorN * (offset - rint(offset));
        const double edge = k_node * sqrt(t0x * t0x + t0y * t0y);
        for (int i = 0; i < 3; ++i)
            eb[EB_DIR + i] = kPhasorN * bd[i];
        eb[EB_PHASE] =
            part + (cls == BEAM_TRAPEZOID || cls == BEAM_VERTICES ? kPhasorN / 4 : 0) + kNodeMagic;
        const double sing = eps_mixed * edge;
        // BEAM_SLOPES: max(|A|, |B|) in nodes above which some phase exceeds 0.25 rad
        const double lim = cls == BEAM_SLOPES
                               ? (kPhasorN * kInvTwoPi * kSmallPhaseMixed / kSmallPhase) * h[H_PHB]
                               : fmax(sing, kLookStep);
        eb[EB_LIM] = pack_floats((float)lim, (float)sing);
        // F of a beam with a value that is not finite is NaN in every direction: the
        // FP64 phases see to that by themselves, the mixed ones lose it as words
        const double inverse = finite == 1.0 ? 1.0 / scale : __builtin_nan("");
        eb[EB_SCALE] = pack_floats((float)(scale / s64), (float)inverse);
        eb[EB_KIND] = pack_words(nv + BEAM_CLASS * cls, 2 * cls64 + (ext ? 1 : 0));
        eb[EB_VOFF] = __builtin_bit_cast(double, v0);
        eb[EB_PHASE64] = part + (cls64 == BEAM_TRAPEZOID ? kPhasorN / 4 : 0);
        eb[EB_S64] = s64;
        // every vertex phase within 1e-3 rad: half of edge 0's step is within that,
        // or the projections within the bound below (see H_PHB)
        const double small = 1.02 * kSmallPhase * (kPhasorN * kInvTwoPi);
        eb[EB_LOOK64] = cls64 == BEAM_VERTICES   ? h[H_PHB] * kPhasorN
                        : cls64 == BEAM_PARALLEL ? small
                                                 : fmax(eps1 * edge, 2.0 * small);
        eb[EB_SING64] = cls64 == BEAM_VERTICES ? eps1 * k_node * lmax
                        : cls64 == BEAM_TRAPEZOID ? eps1 * edge : 0.0;
        h[H_INV] = inverse;
        if (finite != 1.0)  // not for the spectrum source either
            h[H_A0] = __builtin_inf();
        s_scale[g] = ext ? 0.0 : scale;
        s_s64[g] = s64;
    }
    __syncthreads();
    // the records of the workgroup's beams are contiguous
    for (int i = threadIdx.x; i < count * HDR_STRIDE; i += PACK_THREADS)
        hdr[(size_t)first * HDR_STRIDE + i] = s_h[i];
    // W[m][c] = T0[m] Jp[0][c] + T1[m] Jp[1][c], T the rotation vectors halved
    // (exact): column n of beam c
    const auto rotation = [&](int c, int n, double &wr, double &wi) {
        const int m = n >> 2, col = (n >> 1) & 1;
        const double *v = s_bs + c * 36 + (m < 3 ? 13 + m : 16 + m);  // NT NP nxDT nxDP
        const double t0 = 0.5 * v[0], t1 = 0.5 * v[3], *jp = s_jp[c] + 2 * col;
        wr = t0 * jp[0] + t1 * jp[4];
        wi = t0 * jp[1] + t1 * jp[5];
    };
    for (int i = threadIdx.x; i < count * W64_STRIDE; i += PACK_THREADS) {
        const int c = i / W64_STRIDE, n = i - c * W64_STRIDE;
        double wr, wi;
        rotation(c, n, wr, wi);
        w64[(size_t)first * W64_STRIDE + i] = s_s64[c] * ((n & 1) ? wi : wr);
    }
    // MFMA operand (if there was memory for it), split into three BF16 parts; a shadow
    // beam's is zero: it is summed apart
    if (!wb)
        return;
    for (int i = threadIdx.x; i < count * (2 * WB_COLS); i += PACK_THREADS) {
        const int c = i / (2 * WB_COLS), e = i - c * (2 * WB_COLS);
        const int row = e / WB_COLS, n = e - row * WB_COLS;
        double wr, wi;
        rotation(c, n, wr, wi);
        // rows 0 and 1 multiply Re F and Im F / sqrt(2)
        const double w = s_scale[c] == 0.0 ? 0.0
                                           : s_scale[c] * (row == 0 ? ((n & 1) ? wi : wr)
                                                                    : 1.41421356237309504880 *
                                                                          ((n & 1) ? wr : -wi));
        const uint32_t ph = bf16_bits((float)w);
        const double r1 = w - (double)bf16_value(ph);
        const uint32_t pm = bf16_bits((float)r1);
        const uint32_t pl = bf16_bits((float)(r1 - (double)bf16_value(pm)));
        uint32_t *out = wb + (size_t)first * WB_STRIDE + (size_t)i * WB_WORDS;
        out[0] = out[1] = ph | pm << 16;
        out[2] = ph << 16;
        out[3] = pl << 16;
    }
}

// ---------------------------------------------------------------------------
// The edge sums as the reference has them, for beams of class BEAM_SLOPES and for
// lanes next to a singular edge.  Its two branches (|B| > |A|: sum over edges with
// valid dx, coefficient A + (dy/dx) B, divide by B; otherwise edges with
// valid dy, coefficient A (dx/dy) + B, divide by -A) are evaluated by one
// loop whose operands are selected per lane, so lanes that take different
// branches do not diverge.  complWave is folded into J_phased and the
// small-phase area limit at packing time.
// ---------------------------------------------------------------------------
// A wave-uniform FP64 value kept in scalar registers.  Both edge slopes are
// read as scalars and the per-lane choice is made between registers; without
// this the compiler may select the address per lane instead, turning two
// scalar loads into one vector load on every edge.
__device__ __forceinline__ double uniform_f64(double x)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The edge flags of a vertex, in a scalar register.
__device__ __forceinline__ int vertex_flags(const double *__restrict__ vx, int e)
{
    return __builtin_amdgcn_readfirstlane(low_word(vx[(size_t)e * VX_STRIDE + VX_FLAG]));
}

// Every vertex phase within 1e-3 rad: the cell takes the small-phase moment
// form and its edge sum is not used, so the near-singular edges need not be
// evaluated.  That matters: a beam leaving along the incident direction
// (through parallel facets) meets it with A = B = 0 on the theta = 0 row,
// whose azimuth cells lie in as many different waves.
__device__ __forceinline__ bool all_phases_small(const double *__restrict__ vtx, int nv, double A,
                                                 double B, double limit = kSmallPhase)
{
    bool small = true;
    for (int e = 0; e < nv; ++e) {
        const double *v = vtx + (size_t)e * VTX_STRIDE;
        small = small && __builtin_fabs(__builtin_fma(A, v[V_KX], B * v[V_KY])) <= limit;
    }
    return small;
}

// A lane holds its direction d as 1024 d, so that phases come out in nodes.
constexpr double kNode = 1.0 / kPhasorN;
static_assert(kPhasorN == kTabN, "both precisions count phases in the same nodes");

// Nodes of a radian, and a node in radians.
constexpr double kNodes = kPhasorN * kInvTwoPi, kPerNode = 6.28318530717958647693 / kPhasorN;

// The sum over the edges as the reference's two branches have it, in FP64: G = sum
// (e^{i phi_{e+1}} - e^{i phi_e}) / c_e, where c = A + (dy/dx) B (|B| > |A|) or A
// (dx/dy) + B (otherwise), and edges with |c| <= limit are left to
// singular_edges_f64.  A, B in any unit (that of c and limit); `place` gives a
// vertex's place between nodes and table entry.  NV > 0 is the vertex count known
// at compile time: every vertex's table read is issued before the first is used.
// No branch for the singular edges in here: one after every edge, and the flags read
// for it, kept an edge's loads and instructions from passing those of the one
// before.  4,000 beams with slopes of their own on 541 x 96 directions: 2.05 ms with
// these, 1.76 without (of five vertices, one edge a turn: 3.41, now 2.06; the former
// kernel, which rotated each beam and kept fewer sums, 1.60 to 1.77 and 2.1 to
// 2.2).  An invalid edge's stored slope makes its reciprocal vanish.  Returns the
// lanes with an edge within the limit.
template <int NV, typename Place>
__device__ __forceinline__ uint64_t edges_f64(const double *__restrict__ vtx, int nv, double A,
                                              double B, bool useB, double limit, Place place,
                                              double &sr, double &si)
{
    uint64_t near = 0;
    sr = si = 0.0;
    const auto edge = [&](int e, double sp, double cp, double sn, double cn) {
        const double *v = vtx + e * VTX_STRIDE;
        const double cx = __builtin_fma(uniform_f64(v[V_SYX]), B, A),
                     cy = __builtin_fma(uniform_f64(v[V_SXY]), A, B);
        const double cc = useB ? cx : cy;
        const bool big = __builtin_fabs(cc) > limit;
        const double inv = big ? rcp_f64_fast(cc) : 0.0;
        near |= __builtin_amdgcn_ballot_w64(!big);
        sr = __builtin_fma(cn - cp, inv, sr);
        si = __builtin_fma(sn - sp, inv, si);
    };
    if constexpr (NV > 0) {
        double r[NV], sv[NV], cv[NV];
        double2 t[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v)
            place(v, r[v], t[v]);
#pragma unroll
        for (int v = 0; v < NV; ++v)
            node_finish(r[v], t[v], sv[v], cv[v]);
#pragma unroll
        for (int e = 0; e < NV; ++e) {
            const int f = e + 1 < NV ? e + 1 : 0;
            edge(e, sv[e], cv[e], sv[f], cv[f]);
        }
    } else {  // two edges at a time (the compiler does not unroll loops that vote)
        const auto vertex = [&](int v, double &sn, double &cs) {
            double r;
            double2 t;
            place(v, r, t);
            node_finish(r, t, sn, cs);
        };
        double s0, c0, sn, cn;
        vertex(0, s0, c0);
        double sp = s0, cp = c0;
        int e = 0;
        for (; e + 2 < nv; e += 2) {
            vertex(e + 1, sn, cn);
            edge(e, sp, cp, sn, cn);
            vertex(e + 2, sp, cp);
            edge(e + 1, sn, cn, sp, cp);
        }
        if (e + 1 < nv) {
            vertex(e + 1, sn, cn);
            edge(e, sp, cp, sn, cn);
            sp = sn;
            cp = cn;
        }
        edge(nv - 1, sp, cp, s0, c0);
    }
    return near;
}

// What the edges within the limit add to the sum of edges_f64, in a lane that has
// one: the exact half-angle form, which reads the next vertex's phasor only where the
// edge is longer than it serves.  (Edges found by a mask first, theirs alone visited:
// the mask costs the common path registers and 2 to 10 %.)
template <typename Place>
__device__ __forceinline__ void singular_edges_f64(const double *__restrict__ vtx,
                                                   const double *__restrict__ vx, int nv,
                                                   double a, double b, bool useB, double limit,
                                                   double k, Place place,
                                                   double &sr, double &si)
{
    for (int e = 0; e < nv; ++e) {
        const double *v = vtx + e * VTX_STRIDE, *w = vx + e * VX_STRIDE;
        const double cc = useB ? __builtin_fma(uniform_f64(v[V_SYX]), b, a)
                               : __builtin_fma(uniform_f64(v[V_SXY]), a, b);
        if (__builtin_fabs(cc) > limit || !(vertex_flags(w, 0) & (useB ? EDGE_VX : EDGE_VY)))
            continue;
        double r, sp, cp;
        double2 t;
        place(e, r, t);
        node_finish(r, t, sp, cp);
        const double dx = uniform_f64(w[VX_DX]), dy = uniform_f64(w[VX_DY]);
        const double delta = useB ? dx : dy, c = kPerNode * cc;
        double sn = sp, cn = cp;
        if (!(__builtin_fabs(k * c * delta) <= kHalfAngle)) {  // (no half-angle form)
            place(e + 1 < nv ? e + 1 : 0, r, t);
            node_finish(r, t, sn, cn);
        }
        const double2 q = stable_edge_quotient(cp, sp, cn, sn, delta, c, k);
        sr = __builtin_fma(kPerNode, q.x, sr);
        si = __builtin_fma(kPerNode, q.y, si);
    }
}

// Aperture integral F(beam, direction) / complWave in FP64 by the reference's
// branches.  k0, k1, k2: 1024 (d - b), d: 1024 times the direction.  Returns
// false when the result is NaN (degenerate beam, skipped).
__device__ __forceinline__ bool aperture_f64(const double *__restrict__ h,
                                             const double *__restrict__ vtx,
                                             const double *__restrict__ vx, int nv, double k0,
                                             double k1, double k2, const double *d,
                                             const double2 *__restrict__ tab, double k,
                                             double eps1, double &fr, double &fi)
{
    // a word of the first, a middle and the last cache line of the vertices (four lie
    // in two or three): they come beside the header, not after it
    const double t0 = vtx[0], t1 = vtx[2 * VTX_STRIDE], t2 = vtx[nv * VTX_STRIDE - 1];
    // the projections A, B of k - k0 = b - d on the aperture axes and psi = d . kc,
    // times 1024 / 2 pi: a vertex's phase in nodes is a k x + b k y + c, psi folded in
    // (the integral is linear in each phasor), as the reference CUDA path does
    // (GpuDiffraction.cu:1110-1122).  The coefficients take the same a, b: rounded
    // apart from the phases they would not cancel with them.
    const double a = -kInvTwoPi * (k0 * h[H_HOR] + k1 * h[H_HOR + 1] + k2 * h[H_HOR + 2]);
    const double b = -kInvTwoPi * (k0 * h[H_VER] + k1 * h[H_VER + 1] + k2 * h[H_VER + 2]);
    double c = kInvTwoPi * (d[0] * h[H_KC] + d[1] * h[H_KC + 1] + d[2] * h[H_KC + 2]);
    // Without its whole turns (exact), so that a vertex's phase, a hundred times
    // smaller then, is rounded that much finer: the rounding stands over an edge's own
    // small step (1 % of the kernel with slopes of their own, 1.76 -> 1.78 ms)
    c = __builtin_fma(-kPhasorN, __builtin_rint(kNode * c), c);
    const bool useB = __builtin_fabs(b) > __builtin_fabs(a);
    asm volatile("" ::"s"(t0), "s"(t1), "s"(t2));
    const auto place = [&](int v, double &r, double2 &t) {
        const double *q = vtx + v * VTX_STRIDE;
        node_reduce(__builtin_fma(a, uniform_f64(q[V_KX]),
                                  __builtin_fma(b, uniform_f64(q[V_KY]), c)),
                    tab, r, t);
    };
    const double limit = kNodes * eps1;
    // the vertex phases one by one only where the beam's bound leaves the
    // small-phase form possible
    const double larger = useB ? b : -a;
    bool small = false;
    if (__builtin_expect(__builtin_fabs(larger) <= kNodes * h[H_PHB], 0))
        small = all_phases_small(vtx, nv, a, b, kNodes * kSmallPhase);
    double sr = 0.0, si = 0.0;
    uint64_t near = 0;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!small) != 0, 1)) {
        if (nv == 4)
            near = edges_f64<4>(vtx, 4, a, b, useB, limit, place, sr, si);
        else if (nv == 3)
            near = edges_f64<3>(vtx, 3, a, b, useB, limit, place, sr, si);
        else
            near = edges_f64<0>(vtx, nv, a, b, useB, limit, place, sr, si);
    }
    if (__builtin_expect(near != 0, 0)) {
        if (__builtin_amdgcn_inverse_ballot_w64(near) && !small)
            singular_edges_f64(vtx, vx, nv, a, b, useB, limit, k, place, sr, si);
    }
    const double nrm = rcp_f64(kPerNode * kPerNode * larger);
    fr = sr * nrm;
    fi = si * nrm;
    if (__builtin_expect(small, 0)) {
        // small-phase moment form (HandlerPO_fast.h:161-216); the area limit
        // is stored divided by complWave
        const double A = kPerNode * a, B = kPerNode * b;
        const double p1 = A * h[H_MOM] + B * h[H_MOM + 1];
        const double p2 = A * A * h[H_MOM + 2] + A * B * h[H_MOM + 3] + B * B * h[H_MOM + 4];
        const double gr = 1.0 - 0.5 * p2, gi = p1;
        const double ar = h[H_AL] * gr - h[H_AL + 1] * gi;
        const double ai = h[H_AL] * gi + h[H_AL + 1] * gr;
        double r, sd, cd;
        double2 t;
        node_reduce(c, tab, r, t);
        node_finish(r, t, sd, cd);
        fr = ar * cd - ai * sd;
        fi = ar * sd + ai * cd;
    }
    return !__builtin_isnan(fr);
}

// ---- polygon classes ------------------------------------------------------
//
// The aperture integral over a polygon with edges t_e, phases phi_v at its
// vertices and phase steps D_e = phi_{e+1} - phi_e is, for ANY direction q,
//   F = -(k / K.q) sum_e (q x t_e) (e^{i phi_{e+1}} - e^{i phi_e}) / D_e,
// K = k (A, B) / k the projected wave vector: the reference's two branches are
// q = y (divide by B, weights dx) and q = x (divide by -A, weights dy).  With q
// = t_0 the weights are constants of the beam, K.q is edge 0's own phase step,
// edge 0 drops out of the sum, and no lane chooses a branch:
//   F = sum_{e>0} w_e (e^{i phi_{e+1}} - e^{i phi_e}) / D_e / D_0.
// Nothing but phases at points of the aperture is needed of the direction, so
// A, B and psi are not formed either: a phase is three FMAs from d - b and a
// packed vector, its constant term the accumulator they start from.  And with an
// edge's middle phase m_e and half step h_e = D_e / 2, (e^{i phi_{e+1}} -
// e^{i phi_e}) / D_e = i e^{i m_e} sin(h_e) / h_e / 2, which does not cancel as
// D_e goes to zero: no edge but edge 0 is ever singular.
//
// An edge parallel to t_0 has no weight, and then the other two edges of a
// quadrilateral have opposite weights; a triangle is the same with that edge
// shrunk to a point (l: the last edge):
//   F = 2 i w_1 (e^{i m_1} sin(h_1) / D_1 - e^{i m_l} sin(h_l) / D_l) / D_0,
// and for a parallelogram with centre phase m
//   F = -4 w_1 e^{i m} sin(h_0) sin(h_1) / (D_0 D_1).
// The constants go into the packed W.  A traced column's beams are 0.32
// parallelograms, 0.61 trapezoids and triangles; the 8-column aggregate's 0.09
// and 0.63.
//
// FP64: a parallelogram takes 112 vector instructions and a trapezoid 138, the
// sum into G included, where the reference's branches (A, B, psi, two
// coefficients and a select per edge, four phasors with an extra constant and a
// longer polynomial each) took 214; other polygons the sum over their vertices with
// the reference's weights.  35,800 beams of 2,000-15,000 an orientation on 541 x 96
// directions: 8.65 ms against 12.7 for the kernel, which the vector ALU bounds (144
// instructions a beam and wave over 139,000 beams; four waves a SIMD leave it 84 %
// busy).  The error against extended precision is 0.04 to 0.4 of the branches' on the
// mean over draws, workload by workload, and single draws go either way (30 fixed
// orientations on 91 x 16 directions: 0.39 on the mean, 2.8 at the most).

// 1/x to full FP64 precision from the hardware estimate e (1 + e + e^2).
__device__ __forceinline__ double rcp_f64_cubic(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(__builtin_fma(e, e, e), r, r);
}

// F' = sum over the edges of (dx or dy) (e^{i phi_{e+1}} - e^{i phi_e}) / D_e, over
// b or -a: a polygon that is neither triangle, trapezoid nor parallelogram, by the
// reference's weights.  `reach` is |b| or |a|, `step` the least |D_e|.
template <int NV>
__device__ __forceinline__ void aperture_vertices_f64(const double *__restrict__ h,
                                                      const double *__restrict__ vtx,
                                                      const double *__restrict__ vx, int nv,
                                                      double k0, double k1, double k2,
                                                      const double *d,
                                                      const double2 *__restrict__ tab,
                                                      double &fr, double &fi, double &reach,
                                                      double &step)
{
    const double A = k0 * h[H_HOR] + k1 * h[H_HOR + 1] + k2 * h[H_HOR + 2];
    const double B = k0 * h[H_VER] + k1 * h[H_VER + 1] + k2 * h[H_VER + 2];
    const double a = -kInvTwoPi * A, b = -kInvTwoPi * B;
    const double c = kInvTwoPi * (d[0] * h[H_KC] + d[1] * h[H_KC + 1] + d[2] * h[H_KC + 2]);
    // the weights over K.q: dx / b, or -dy / a
    const bool useB = __builtin_fabs(B) > __builtin_fabs(A);
    const double over = rcp_f64_cubic(useB ? b : -a);
    const double ux = useB ? over : 0.0, uy = useB ? 0.0 : over;
    reach = __builtin_fabs(useB ? B : A);
    const auto vertex = [&](int v, double &p, double &sn, double &cs) {
        const double *q = vtx + v * VTX_STRIDE;
        p = __builtin_fma(a, q[V_KX], __builtin_fma(b, q[V_KY], c));
        double r;
        double2 e;
        node_reduce(p, tab, r, e);
        node_finish(r, e, sn, cs);
    };
    // edge e, from a vertex (phase, sine and cosine p, sp, cp) to the next (n, sn, cn)
    double sr = 0.0, si = 0.0;
    step = __builtin_inf();
    const auto edge = [&](int e, double p, double sp, double cp, double n, double sn, double cn) {
        const double dx = uniform_f64(vx[e * VX_STRIDE + VX_DX]),
                     dy = uniform_f64(vx[e * VX_STRIDE + VX_DY]);
        const double D = n - p;
        const double w = __builtin_fma(dy, uy, dx * ux) * rcp_f64_cubic(D);
        sr = __builtin_fma(cn - cp, w, sr);
        si = __builtin_fma(sn - sp, w, si);
        step = __builtin_fmin(step, __builtin_fabs(D));
    };
    double p0, s0, c0;
    vertex(0, p0, s0, c0);
    double p = p0, sp = s0, cp = c0, n, sn, cn;
    const int last = (NV > 0 ? NV : nv) - 1;
    int e = 0;
    // two edges at a time (the compiler does not unroll loops that read lanes)
#pragma unroll
    for (; e + 2 <= last; e += 2) {
        vertex(e + 1, n, sn, cn);
        edge(e, p, sp, cp, n, sn, cn);
        vertex(e + 2, p, sp, cp);
        edge(e + 1, n, sn, cn, p, sp, cp);
    }
    if (e < last) {
        vertex(last, n, sn, cn);
        edge(e, p, sp, cp, n, sn, cn);
        edge(last, n, sn, cn, p0, s0, c0);
    } else {
        edge(last, p, sp, cp, p0, s0, c0);
    }
    fr = sr;
    fi = si;
}

// F' = F / complWave / s of a beam in a direction, s its EB_S64.  Returns the
// lanes (a mask) whose F is NaN: there the beam does not count (HandlerPO.cpp:2742).
// Lane conditions are kept as scalar masks: as bools they would cross the
// blocks in vector registers.
__device__ __forceinline__ uint64_t aperture_any_f64(const double *eb, const double *__restrict__ h,
                                                 const double *__restrict__ vtxs,
                                                 const double *__restrict__ vxs, const double *d,
                                                 const double2 *__restrict__ tab, double k,
                                                 double eps1, double &fr, double &fi)
{
    const int cls = high_word(eb[EB_KIND]) >> 1;
    const int nv = low_word(eb[EB_KIND]) & BEAM_NV;
    const int64_t v0 = __builtin_bit_cast(int64_t, eb[EB_VOFF]);
    const double *vtx = vtxs + (size_t)v0 * VTX_STRIDE, *vx = vxs + (size_t)v0 * VX_STRIDE;
    const double k0 = d[0] - eb[EB_DIR], k1 = d[1] - eb[EB_DIR + 1], k2 = d[2] - eb[EB_DIR + 2];
    const auto half = [&](const double *q) {
        return __builtin_fma(k2, q[2], __builtin_fma(k1, q[1], k0 * q[0]));
    };
    const auto phase = [&](const double *q) {
        return __builtin_fma(k2, q[2], __builtin_fma(k1, q[1], __builtin_fma(k0, q[0],
                                                                             eb[EB_PHASE64])));
    };
    const double *q = eb + EB_Q;
    uint64_t look = 0, general = 0, dead = 0;
    // edge 0's step (the least step), and the divisor, which may be zero without it
    double step = 1.0, div = 1.0;
    if (cls == BEAM_TRAPEZOID) {
        const double m1 = phase(q), h1 = half(q + 3), m3 = phase(q + 6), h3 = half(q + 9);
        double rm1, rh1, rm3, rh3;
        double2 em1, eh1, em3, eh3;
        node_reduce(m1, tab, rm1, em1);
        node_reduce(h1, tab, rh1, eh1);
        node_reduce(m3, tab, rm3, em3);
        node_reduce(h3, tab, rh3, eh3);
        step = (m1 - m3) - (h1 + h3);
        div = h1 * h3 * step;
        const double r = rcp_f64_cubic(div);
        const double q1 = node_sine(rh1, eh1) * h3, q3 = node_sine(rh3, eh3) * h1;
        double s1, c1, s3, c3;
        node_finish(rm1, em1, s1, c1);
        node_finish(rm3, em3, s3, c3);
        fr = __builtin_fma(q1, c1, -(q3 * c3)) * r;
        fi = __builtin_fma(q1, s1, -(q3 * s3)) * r;
        look = __builtin_amdgcn_ballot_w64(!(__builtin_fabs(step) >= eb[EB_LOOK64])) |
               __builtin_amdgcn_ballot_w64(div == 0.0);
    } else if (cls == BEAM_PARALLEL) {
        const double m = phase(q), h1 = half(q + 6);
        step = half(q + 3);
        double rm, r0, r1;
        double2 em, e0, e1;
        node_reduce(m, tab, rm, em);
        node_reduce(step, tab, r0, e0);
        node_reduce(h1, tab, r1, e1);
        div = step * h1;
        const double f = node_sine(r0, e0) * node_sine(r1, e1) * rcp_f64_cubic(div);
        double s, c;
        node_finish(rm, em, s, c);
        fr = c * f;
        fi = s * f;
        look = __builtin_amdgcn_ballot_w64(!(__builtin_fabs(step) >= eb[EB_LOOK64])) |
               __builtin_amdgcn_ballot_w64(div == 0.0);
    } else if (cls == BEAM_VERTICES) {
        double reach;
        if (nv == 4)
            aperture_vertices_f64<4>(h, vtx, vx, 4, k0, k1, k2, d, tab, fr, fi, reach, step);
        else
            aperture_vertices_f64<0>(h, vtx, vx, nv, k0, k1, k2, d, tab, fr, fi, reach, step);
        look = __builtin_amdgcn_ballot_w64(!(reach > eb[EB_LOOK64])) |
               __builtin_amdgcn_ballot_w64(!(step > eb[EB_SING64]));
    } else {
        general = ~0ull;
    }
    // next to a singular edge, and where every phase is small: the branches
    if (__builtin_expect(look != 0, 0)) {
        // a word of each cache line that the branches read of the polygon, so that
        // they come together and not one after the other
        const double t0 = vtx[0], t1 = vtx[2 * VTX_STRIDE], t2 = vtx[nv * VTX_STRIDE - 1];
        const double t3 = vx[0], t4 = vx[2 * VX_STRIDE], t5 = vx[nv * VX_STRIDE - 1];
        asm volatile("" ::"s"(t0), "s"(t1), "s"(t2), "s"(t3), "s"(t4), "s"(t5));
        const double A = -kNode * (k0 * h[H_HOR] + k1 * h[H_HOR + 1] + k2 * h[H_HOR + 2]);
        const double B = -kNode * (k0 * h[H_VER] + k1 * h[H_VER + 1] + k2 * h[H_VER + 2]);
        const bool leaves = !(__builtin_fabs(step) > eb[EB_SING64]) || div == 0.0 ||
                            all_phases_small(vtx, nv, A, B);
        general = look & __builtin_amdgcn_ballot_w64(leaves);
    }
    if (__builtin_expect(general != 0, 0)) {
        bool ok = true;
        if (__builtin_amdgcn_inverse_ballot_w64(general)) {
            ok = aperture_f64(h, vtx, vx, nv, k0, k1, k2, d, tab, k, eps1, fr, fi);
            if (cls != BEAM_SLOPES) {  // whose EB_S64 is 1
                const double inv = rcp_f64(eb[EB_S64]);
                fr *= inv;
                fi *= inv;
            }
        }
        dead = __builtin_amdgcn_ballot_w64(!ok);
    }
    return dead;
}

// G += F' W: entry 4m + 2c + r of G and of W (po_layout.h).
template <typename T>
__device__ __forceinline__ void add_rotated(const double *__restrict__ w, T fr, T fi, T *g)
{
#pragma unroll
    for (int n = 0; n < W64_STRIDE; n += 2) {
        const T wr = (T)w[n], wi = (T)w[n + 1];
        g[n] = fr * wr + (g[n] - fi * wi);
        g[n + 1] = fr * wi + (g[n + 1] + fi * wr);
    }
}

// The Jones sum of a lane from its G: J[i][c] = sum_m u_i[m] G[m][c]; entry m of u0,
// u1 at m * ld.
template <typename T>
__device__ __forceinline__ void add_jones(const T *g, const T *u, size_t ld, T *j)
{
#pragma unroll
    for (int m = 0; m < 12; ++m) {
        const T um = u[m * ld];
        for (int n = 0; n < 4; ++n)
            j[4 * (m / 6) + n] = um * g[4 * (m % 6) + n] + j[4 * (m / 6) + n];
    }
}

// ---- mixed precision ----------------------------------------------------
//
// The polygon classes above, with phases in fixed-point nodes (the constant term
// of a phase carries the offset kNodeMagic) and FP32 phasors.  Trapezoids take 60
// and parallelograms 40 vector instructions, where the reference's branches (A,
// B, psi, two FP64 coefficients and a select per edge, an FP64 reduction per
// vertex) took 109, and other quadrilaterals 100 (137,000 beams of 2,000-15,000
// an orientation on 541 x 96 directions: 16.8 ms against 27.3 for the kernel,
// contraction included).  From five vertices on (shadow beams, 4 to 15 in 100
// others) the weights are the reference's dx or dy, by the larger of |A| and |B|,
// since one edge's own step is too often small against K there.
//
// Lanes where D_0 is small leave the sums: fix_lanes below.  Forms that were
// shorter and lost precision: one coefficient per vertex, X_v / (D_{v-1} D_v)
// (twice the error: its coefficients multiply phasors, not differences), and the
// sum over edge 0 on phasor differences (1.3 times the error of the branches).

// The moment form: F of a cell whose vertex phases are all within
// kSmallPhaseMixed: <e^{i phi}> = sum_n i^n <phi^n> / n! to
// fifth order, times the area limit and e^{i psi}, and times scale (in FP64: a
// forward peak is all in such a value).  Returns the real part and the imaginary
// part / sqrt(2).
__device__ __forceinline__ void moments_mixed(const double *__restrict__ h, double A, double B,
                                              double psi, double scale,
                                              const PhasorNode *__restrict__ tab,
                                              float &out_r, float &out_s)
{
    const double A2 = A * A, B2 = B * B, AB = A * B;
    const double *c3 = h + H_MOM3, *c4 = h + H_MOM4, *c5 = h + H_MOM5;
    const double p1 = A * h[H_MOM] + B * h[H_MOM + 1];
    const double p2 = A2 * h[H_MOM + 2] + AB * h[H_MOM + 3] + B2 * h[H_MOM + 4];
    const double q3 = B * (B2 * c3[0] + AB * c3[1]) + A * (AB * c3[2] + A2 * c3[3]);
    const double q4 =
        B2 * (B2 * c4[0] + AB * c4[1]) + A2 * (B2 * c4[2] + AB * c4[3] + A2 * c4[4]);
    const double A3 = A * A2, B3 = B * B2;
    const double q5 = B3 * (B2 * c5[0] + AB * c5[1] + A2 * c5[2]) +
                      A3 * (B2 * c5[3] + AB * c5[4] + A2 * c5[5]);
    const double gr = 1.0 - 0.5 * p2 + q4, gi = p1 - q3 + q5;
    const float ar = (float)((h[H_AL] * gr - h[H_AL + 1] * gi) * scale);
    const float ai = (float)((h[H_AL] * gi + h[H_AL + 1] * gr) * scale);
    float c, s;
    phasor_rad(psi, tab, c, s);
    out_r = __builtin_fmaf(-ai * kSqrt2, s, ar * c);
    out_s = __builtin_fmaf(ar, s, ai * kInvSqrt2 * c);
}

// The edge sum over the reference's branches, as the ABI's slopes and flags
// define it: beams of class BEAM_SLOPES and BEAM_FAR, and single lanes of other
// beams next to a singular edge.  As edges_f64, with `word` giving a vertex's
// phase word; the edge coefficient is cancellation-prone and stays in FP64.
template <int NV, typename Word>
__device__ __forceinline__ uint64_t edges_mixed(const double *__restrict__ vtx, int nv, double A,
                                                double B, bool useB, double limit,
                                                const PhasorNode *__restrict__ tab, Word word,
                                                float &sr, float &ss)
{
    uint64_t near = 0;
    sr = ss = 0.0f;
    const auto edge = [&](int e, float cp, float sp, float cn, float sn) {
        const double *v = vtx + e * VTX_STRIDE;
        const double cx = __builtin_fma(uniform_f64(v[V_SYX]), B, A),
                     cy = __builtin_fma(uniform_f64(v[V_SXY]), A, B);
        const double cc = useB ? cx : cy;
        const bool big = __builtin_fabs(cc) > limit;
        const float r = __builtin_amdgcn_rcpf((float)cc);
        const float inv = big ? r : 0.0f;
        near |= __builtin_amdgcn_ballot_w64(!big);
        sr = __builtin_fmaf(cn - cp, inv, sr);
        ss = __builtin_fmaf(sn - sp, inv, ss);
    };
    if constexpr (NV > 0) {
        float cv[NV], sv[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const uint32_t u = word(v);
            phasor_finish(u, phasor_read(u, tab), cv[v], sv[v]);
        }
#pragma unroll
        for (int e = 0; e < NV; ++e) {
            const int f = e + 1 < NV ? e + 1 : 0;
            edge(e, cv[e], sv[e], cv[f], sv[f]);
        }
    } else {  // two edges at a time
        const auto vertex = [&](int v, float &cs, float &sn) {
            const uint32_t u = word(v);
            phasor_finish(u, phasor_read(u, tab), cs, sn);
        };
        float c0, s0, cn, sn;
        vertex(0, c0, s0);
        float cp = c0, sp = s0;
        int e = 0;
        for (; e + 2 < nv; e += 2) {
            vertex(e + 1, cn, sn);
            edge(e, cp, sp, cn, sn);
            vertex(e + 2, cp, sp);
            edge(e + 1, cn, sn, cp, sp);
        }
        if (e + 1 < nv) {
            vertex(e + 1, cn, sn);
            edge(e, cp, sp, cn, sn);
            cp = cn;
            sp = sn;
        }
        edge(nv - 1, cp, sp, c0, s0);
    }
    return near;
}

// As singular_edges_f64, a and b in nodes.
template <typename Word>
__device__ __forceinline__ void singular_edges_mixed(const double *__restrict__ vtx,
                                                     const double *__restrict__ vx, int nv,
                                                     double a, double b, bool useB, double limit,
                                                     double k,
                                                     const PhasorNode *__restrict__ tab,
                                                     Word word, float &sr, float &ss)
{
    for (int e = 0; e < nv; ++e) {
        const double *v = vtx + e * VTX_STRIDE, *w = vx + e * VX_STRIDE;
        const double cc = useB ? __builtin_fma(uniform_f64(v[V_SYX]), b, a)
                               : __builtin_fma(uniform_f64(v[V_SXY]), a, b);
        if (__builtin_fabs(cc) > limit || !(vertex_flags(w, 0) & (useB ? EDGE_VX : EDGE_VY)))
            continue;
        float cp, sp;
        uint32_t u = word(e);
        phasor_finish(u, phasor_read(u, tab), cp, sp);
        const double dx = uniform_f64(w[VX_DX]), dy = uniform_f64(w[VX_DY]);
        const double delta = useB ? dx : dy, c = kPerNode * cc;
        float cn = cp, sn = sp;
        if (!(__builtin_fabs(k * c * delta) <= kHalfAngle)) {  // (no half-angle form)
            u = word(e + 1 < nv ? e + 1 : 0);
            phasor_finish(u, phasor_read(u, tab), cn, sn);
        }
        const double2 q = stable_edge_quotient((double)cp, (double)(sp * kSqrt2), (double)cn,
                                               (double)(sn * kSqrt2), delta, c, k);
        sr += (float)(kPerNode * q.x);
        ss += (float)(kPerNode * q.y * (double)kInvSqrt2);
    }
}

// F' of the lanes that the formulas over edge 0 leave: those with small phases
// (`maybe` those to be tested for it) by the moments, those next to a singular
// edge, and every lane of a BEAM_SLOPES or BEAM_FAR beam, by the reference's
// branches.
__device__ __forceinline__ void fix_lanes(const double *eb, const double *__restrict__ h,
                                          const double *__restrict__ vtx,
                                          const double *__restrict__ vx, int nv, int cls,
                                          const double *d, bool singular, bool maybe,
                                          const PhasorNode *__restrict__ tab, double k,
                                          double eps1, float &out_r, float &out_s)
{
    // A, B: projections of k - k0 = b - d on the aperture axes
    const double k0 = kNode * (eb[EB_DIR] - d[0]), k1 = kNode * (eb[EB_DIR + 1] - d[1]),
                 k2 = kNode * (eb[EB_DIR + 2] - d[2]);
    const double A = k0 * h[H_HOR] + k1 * h[H_HOR + 1] + k2 * h[H_HOR + 2];
    const double B = k0 * h[H_VER] + k1 * h[H_VER + 1] + k2 * h[H_VER + 2];
    const double psi = kNode * (d[0] * h[H_KC] + d[1] * h[H_KC + 1] + d[2] * h[H_KC + 2]);
    bool small = maybe;
    if (cls == BEAM_FAR)  // (the other classes' steps have told)
        small = __builtin_fmax(__builtin_fabs(A), __builtin_fabs(B)) <=
                (kSmallPhaseMixed / kSmallPhase) * h[H_PHB];
    if (cls != BEAM_MOMENTS)
        small = small && all_phases_small(vtx, nv, A, B, kSmallPhaseMixed);
    if (singular && !small) {
        const double a = kNodes * A, b = kNodes * B, c = kNodes * psi;
        const bool useB = __builtin_fabs(b) > __builtin_fabs(a);
        const auto word = [&](int v) {  // of any size: to half a turn first
            const double *q = vtx + v * VTX_STRIDE;
            const double p = __builtin_fma(a, uniform_f64(q[V_KX]),
                                           __builtin_fma(b, uniform_f64(q[V_KY]), c));
            return low_bits(__builtin_fma(-(double)kPhasorN, __builtin_rint(kNode * p), p) +
                            kNodeMagic);
        };
        float sr, ss;
        const uint64_t near = edges_mixed<0>(vtx, nv, a, b, useB, kNodes * eps1, tab, word, sr, ss);
        if (__builtin_amdgcn_inverse_ballot_w64(near))
            singular_edges_mixed(vtx, vx, nv, a, b, useB, kNodes * eps1, k, tab, word, sr, ss);
        const float nrm = __builtin_amdgcn_rcpf((float)(useB ? b : -a)) *
                          ((float)(kNodes * kNodes) * high_float(eb[EB_SCALE]));
        out_r = sr * nrm;
        out_s = ss * nrm;
    }
    if (small)
        moments_mixed(h, A, B, psi, h[H_INV], tab, out_r, out_s);
    if (singular || small) {
        // a NaN F (degenerate polygon) counts as zero
        const bool bad = __builtin_isnan(out_r);
        out_r = bad ? 0.0f : out_r;
        out_s = bad ? 0.0f : out_s;
    }
}

// sin(h) / sqrt(2) / f from the series, for a small half step of f nodes (h rad).
__device__ __forceinline__ float sine_ratio_series(float f)
{
    const float x = (float)(6.28318530717958648 / kPhasorN) * f, z = x * x;
    return (float)(4.44288293815836625 / kPhasorN) *
           __builtin_fmaf(z, __builtin_fmaf(z, 1.0f / 120.0f, -1.0f / 6.0f), 1.0f);
}

// Triangles and trapezoids.
__device__ __forceinline__ void aperture_trapezoid(const double *eb, const double *d,
                                                   const PhasorNode *__restrict__ tab,
                                                   float &out_r, float &out_s,
                                                   uint64_t &singular, uint64_t &maybe)
{
    const double k0 = d[0] - eb[EB_DIR], k1 = d[1] - eb[EB_DIR + 1], k2 = d[2] - eb[EB_DIR + 2];
    const auto phase = [&](const double *q, double c) {
        return __builtin_fma(k2, q[2], __builtin_fma(k1, q[1], __builtin_fma(k0, q[0], c)));
    };
    const double *q = eb + EB_Q;
    const double m1 = phase(q, eb[EB_PHASE]), a1 = phase(q + 3, kNodeMagic);
    const double m3 = phase(q + 6, eb[EB_PHASE]), a3 = phase(q + 9, kNodeMagic);
    const PhasorNode em1 = phasor_read(low_bits(m1), tab), ea1 = phasor_read(low_bits(a1), tab),
                     em3 = phasor_read(low_bits(m3), tab), ea3 = phasor_read(low_bits(a3), tab);
    const double h1 = a1 - kNodeMagic, h3 = a3 - kNodeMagic;
    const float f1 = (float)h1, f3 = (float)h3;
    const float step = (float)((m1 - m3) - (h1 + h3));  // edge 0
    const float r0 = __builtin_amdgcn_rcpf(step);
    float c1, s1, c3, s3;
    phasor_finish(low_bits(m1), em1, c1, s1);
    phasor_finish(low_bits(m3), em3, c3, s3);
    float q1 = sine_finish(low_bits(a1), ea1) * __builtin_amdgcn_rcpf(f1);
    float q3 = sine_finish(low_bits(a3), ea3) * __builtin_amdgcn_rcpf(f3);
    const bool series =
        __builtin_fminf(__builtin_fabsf(f1), __builtin_fabsf(f3)) < kSeriesStep;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(series) != 0, 0)) {
        q1 = __builtin_fabsf(f1) < kSeriesStep ? sine_ratio_series(f1) : q1;
        q3 = __builtin_fabsf(f3) < kSeriesStep ? sine_ratio_series(f3) : q3;
    }
    out_r = __builtin_fmaf(q1, c1, -(q3 * c3)) * r0;
    out_s = __builtin_fmaf(q1, s1, -(q3 * s3)) * r0;
    const bool look = !(__builtin_fabsf(step) >= low_float(eb[EB_LIM]));
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(look) != 0, 0)) {
        singular =
            __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(step) >= high_float(eb[EB_LIM])));
        maybe = __builtin_amdgcn_ballot_w64(
            look &&
            __builtin_fmaxf(__builtin_fabsf(f1), __builtin_fabsf(f3)) <= (float)kLookStep);
    }
}

// Parallelograms.
__device__ __forceinline__ void aperture_parallelogram(const double *eb, const double *d,
                                                       const PhasorNode *__restrict__ tab,
                                                       float &out_r, float &out_s)
{
    const double k0 = d[0] - eb[EB_DIR], k1 = d[1] - eb[EB_DIR + 1], k2 = d[2] - eb[EB_DIR + 2];
    const auto phase = [&](const double *q, double c) {
        return __builtin_fma(k2, q[2], __builtin_fma(k1, q[1], __builtin_fma(k0, q[0], c)));
    };
    const double m = phase(eb + EB_Q, eb[EB_PHASE]);
    const double a0 = phase(eb + EB_Q + 3, kNodeMagic), a1 = phase(eb + EB_Q + 6, kNodeMagic);
    const PhasorNode em = phasor_read(low_bits(m), tab), e0 = phasor_read(low_bits(a0), tab),
                     e1 = phasor_read(low_bits(a1), tab);
    const float f0 = (float)(a0 - kNodeMagic), f1 = (float)(a1 - kNodeMagic);
    float c, s;
    phasor_finish(low_bits(m), em, c, s);
    const float s0 = sine_finish(low_bits(a0), e0), s1 = sine_finish(low_bits(a1), e1);
    float q = s0 * s1 * __builtin_amdgcn_rcpf(f0 * f1);
    const bool series =
        __builtin_fminf(__builtin_fabsf(f0), __builtin_fabsf(f1)) < kSeriesStep;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(series) != 0, 0)) {
        if (series) {
            const float q0 = __builtin_fabsf(f0) < kSeriesStep
                                 ? sine_ratio_series(f0)
                                 : s0 * __builtin_amdgcn_rcpf(f0);
            const float q1 = __builtin_fabsf(f1) < kSeriesStep
                                 ? sine_ratio_series(f1)
                                 : s1 * __builtin_amdgcn_rcpf(f1);
            q = q0 * q1;
        }
    }
    out_r = q * c;
    out_s = q * s;
}

// One edge's (cos, sin / sqrt 2) of the middle phase and sin / sqrt(2) / f of its
// half step, f nodes, from the phases p, n (with kNodeMagic) of its ends.
__device__ __forceinline__ void edge_terms(double p, double n,
                                           const PhasorNode *__restrict__ tab, float &c,
                                           float &s, float &q, float &f)
{
    const double m = 0.5 * (p + n), a = __builtin_fma(0.5, n - p, kNodeMagic);
    const PhasorNode em = phasor_read(low_bits(m), tab), ea = phasor_read(low_bits(a), tab);
    f = (float)(a - kNodeMagic);
    phasor_finish(low_bits(m), em, c, s);
    q = sine_finish(low_bits(a), ea) * __builtin_amdgcn_rcpf(f);
    const bool series = __builtin_fabsf(f) < kSeriesStep;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(series) != 0, 0))
        q = series ? sine_ratio_series(f) : q;
}

// The projections -A / 2 pi, -B / 2 pi ... of d - b for the classes with vertices:
// a vertex's phase is a k x + b k y + c.
struct Projection {
    double a, b, c;
};
__device__ __forceinline__ Projection project(const double *eb, const double *d)
{
    const double k0 = d[0] - eb[EB_DIR], k1 = d[1] - eb[EB_DIR + 1], k2 = d[2] - eb[EB_DIR + 2];
    const double *q = eb + EB_Q;
    return {__builtin_fma(k2, q[2], __builtin_fma(k1, q[1], k0 * q[0])),
            __builtin_fma(k2, q[5], __builtin_fma(k1, q[4], k0 * q[3])),
            __builtin_fma(k2, q[8], __builtin_fma(k1, q[7], __builtin_fma(k0, q[6],
                                                                          eb[EB_PHASE])))};
}
__device__ __forceinline__ double vertex_phase(const Projection &p, const double *v)
{
    return __builtin_fma(p.a, v[V_KX], __builtin_fma(p.b, v[V_KY], p.c));
}

// The sum over edge 0 for the other quadrilaterals.
__device__ __forceinline__ void aperture_quad(const double *eb, const double *__restrict__ vtx,
                                              const double *__restrict__ vx, const double *d,
                                              const PhasorNode *__restrict__ tab, float &out_r,
                                              float &out_s, uint64_t &singular, uint64_t &maybe)
{
    const Projection p = project(eb, d);
    double ph[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        ph[v] = vertex_phase(p, vtx + v * VTX_STRIDE);
    const float step = (float)(ph[1] - ph[0]);
    float sr = 0.0f, ss = 0.0f, legs = 0.0f;
#pragma unroll
    for (int e = 1; e < 4; ++e) {
        float c, s, q, f;
        edge_terms(ph[e], ph[(e + 1) % 4], tab, c, s, q, f);
        const float coef = q * low_float(vx[e * VX_STRIDE + VX_W]);
        sr = __builtin_fmaf(c, coef, sr);
        ss = __builtin_fmaf(s, coef, ss);
        legs = __builtin_fmaxf(legs, __builtin_fabsf(f));
    }
    const float r0 = __builtin_amdgcn_rcpf(step);
    out_r = sr * r0;
    out_s = ss * r0;
    singular = __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(step) >= high_float(eb[EB_LIM])));
    maybe = __builtin_amdgcn_ballot_w64(__builtin_fmaxf(legs, __builtin_fabsf(step)) <=
                                        (float)kLookStep);
}

// Five vertices and more, one at a time, with the reference's weights.
__device__ __forceinline__ void aperture_loop(const double *eb, const double *__restrict__ vtx,
                                              const double *__restrict__ vx, int nv,
                                              const double *d,
                                              const PhasorNode *__restrict__ tab, float &out_r,
                                              float &out_s, uint64_t &maybe)
{
    const Projection p = project(eb, d);
    const bool useB = __builtin_fabs(p.b) > __builtin_fabs(p.a);
    float sr = 0.0f, ss = 0.0f, steps = 0.0f;
    const auto edge = [&](int e, double from, double to) {
        const double w = vx[e * VX_STRIDE + VX_W];
        const float wx = low_float(w), wy = high_float(w);
        float c, s, ratio, f;
        edge_terms(from, to, tab, c, s, ratio, f);
        const float coef = ratio * (useB ? wx : wy);
        sr = __builtin_fmaf(c, coef, sr);
        ss = __builtin_fmaf(s, coef, ss);
        steps = __builtin_fmaxf(steps, __builtin_fabsf(f));
    };
    // two edges at a time (the compiler does not unroll loops that vote)
    const double p0 = vertex_phase(p, vtx);
    double from = p0;
    int e = 0;
    for (; e + 2 < nv; e += 2) {
        const double mid = vertex_phase(p, vtx + (e + 1) * VTX_STRIDE);
        edge(e, from, mid);
        from = vertex_phase(p, vtx + (e + 2) * VTX_STRIDE);
        edge(e + 1, mid, from);
    }
    if (e + 1 < nv) {
        const double mid = vertex_phase(p, vtx + (e + 1) * VTX_STRIDE);
        edge(e, from, mid);
        from = mid;
    }
    edge(nv - 1, from, p0);
    const float r = __builtin_amdgcn_rcpf((float)(useB ? p.b : p.a));
    out_r = sr * r;
    out_s = ss * r;
    maybe = __builtin_amdgcn_ballot_w64(steps <= (float)kLookStep);
}

// The edge sum with the slopes as given, for phases within the fixed-point range
// (BEAM_SLOPES).  Nothing of the header is read on the way: with it, every vertex's
// phase tested for the moments, and a branch and flags for each edge, a beam waited
// for load after load (4,000 beams on 541 x 96 directions: 1.73 ms, now 0.98; on
// the vector ALU 1.59, now 0.97; the former kernel 1.01 and 0.95).  Lanes with a
// singular edge, or phases that may all be small, go to fix_lanes.
__device__ __forceinline__ void aperture_slopes(const double *eb, const double *__restrict__ vtx,
                                                int nv, const double *d,
                                                const PhasorNode *__restrict__ tab, double eps1,
                                                float &out_r, float &out_s, uint64_t &singular,
                                                uint64_t &maybe)
{
    const Projection p = project(eb, d);
    const bool useB = __builtin_fabs(p.b) > __builtin_fabs(p.a);
    const auto word = [&](int v) { return low_bits(vertex_phase(p, vtx + v * VTX_STRIDE)); };
    float sr, ss;
    if (nv == 4)
        singular = edges_mixed<4>(vtx, 4, p.a, p.b, useB, kNodes * eps1, tab, word, sr, ss);
    else if (nv == 3)
        singular = edges_mixed<3>(vtx, 3, p.a, p.b, useB, kNodes * eps1, tab, word, sr, ss);
    else
        singular = edges_mixed<0>(vtx, nv, p.a, p.b, useB, kNodes * eps1, tab, word, sr, ss);
    const float q = (float)(useB ? p.b : -p.a);
    const float nrm = __builtin_amdgcn_rcpf(q) * (float)(kNodes * kNodes);
    out_r = sr * nrm;
    out_s = ss * nrm;
    maybe = __builtin_amdgcn_ballot_w64(__builtin_fabsf(q) <= low_float(eb[EB_LIM]));
}

// F' = F / complWave / s of a beam in a direction, s = 1 / the second half of its
// EB_SCALE, mixed precision: FP64 phases and moments, FP32 phasors and sums.  eb: the
// beam's record (in registers).  Returns the real part and the imaginary part /
// sqrt(2).
__device__ __forceinline__ void aperture_mixed(const double *eb, const double *__restrict__ h,
                                               const double *__restrict__ vtxs,
                                               const double *__restrict__ vxs, const double *d,
                                               const PhasorNode *__restrict__ tab, double k,
                                               double eps1, float &out_r, float &out_s)
{
    const int kind = low_word(eb[EB_KIND]);
    const int nv = kind & BEAM_NV, cls = kind / BEAM_CLASS;
    const int64_t v0 = __builtin_bit_cast(int64_t, eb[EB_VOFF]);
    const double *vtx = vtxs + (size_t)v0 * VTX_STRIDE, *vx = vxs + (size_t)v0 * VX_STRIDE;
    uint64_t singular = 0, maybe = 0;  // lanes
    out_r = out_s = 0.0f;
    if (cls == BEAM_TRAPEZOID) {
        aperture_trapezoid(eb, d, tab, out_r, out_s, singular, maybe);
    } else if (cls == BEAM_PARALLEL) {
        aperture_parallelogram(eb, d, tab, out_r, out_s);
    } else if (cls == BEAM_VERTICES) {
        if (nv == 4)
            aperture_quad(eb, vtx, vx, d, tab, out_r, out_s, singular, maybe);
        else
            aperture_loop(eb, vtx, vx, nv, d, tab, out_r, out_s, maybe);
    } else if (cls == BEAM_SLOPES) {
        aperture_slopes(eb, vtx, nv, d, tab, eps1, out_r, out_s, singular, maybe);
    } else {
        singular = cls == BEAM_MOMENTS ? 0 : ~0ull;
        maybe = ~0ull;
    }
    if (__builtin_expect((singular | maybe) != 0, 0)) {
        // the branches: a word of each cache line they read of the polygon, so that they
        // come together (3,900 beams on 181 x 48 directions, which wait for the pole
        // rows: 154 us, now 143; asked for with the moments too, those cost 12 % more)
        if (singular) {
            const double t0 = vtx[0], t1 = vtx[2 * VTX_STRIDE], t2 = vtx[nv * VTX_STRIDE - 1];
            const double t3 = vx[0], t4 = vx[2 * VX_STRIDE], t5 = vx[nv * VX_STRIDE - 1];
            const double t6 = h[H_HOR], t7 = h[H_KC];
            asm volatile("" ::"s"(t0), "s"(t1), "s"(t2), "s"(t3), "s"(t4), "s"(t5), "s"(t6),
                         "s"(t7));
        }
        if (__builtin_amdgcn_inverse_ballot_w64(singular | maybe))
            fix_lanes(eb, h, vtx, vx, nv, cls, d, __builtin_amdgcn_inverse_ballot_w64(singular),
                      __builtin_amdgcn_inverse_ballot_w64(maybe), tab, k, eps1, out_r, out_s);
    }
}

// A beam's record in scalar registers.
struct BeamRecord {
    double v[EB_STRIDE];
};
__device__ __forceinline__ BeamRecord load_record(const double *__restrict__ eb)
{
    BeamRecord r;
    for (int i = 0; i < EB_STRIDE; ++i)
        r.v[i] = eb[i];
    return r;
}

// One word of each cache line of a beam's W: brings it into the scalar cache a
// beam ahead.  W (48 registers) and the next record (40) do not fit the scalar
// registers together, so W is read in three parts, each of them waited for; from
// L2 these waits were 6 % of the FP64 kernel's time.  `arrived` ends it.
struct Lines {
    float v[3];
    __device__ __forceinline__ void touch(const double *__restrict__ w)
    {
        for (int i = 0; i < 3; ++i)
            v[i] = *reinterpret_cast<const float *>(w + 8 * i);
    }
    __device__ __forceinline__ void arrived() const
    {
        asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]));
    }
};
static_assert(W64_STRIDE == 24, "three lines of 64 bytes");

// Adds F R Jp to j[8], w the beam's rotation data, u (entry m at m * ld) the lane's
// rotation vectors u0, u1; a loop, to hold few registers.
template <typename T>
__device__ __forceinline__ void rotate_add(const double *__restrict__ w, const T *u, size_t ld,
                                           T fr, T fi, T *j)
{
    T q[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // R Jp
#pragma unroll 1
    for (int m = 0; m < 6; ++m) {
        const T u0 = u[m * ld], u1 = u[(6 + m) * ld];
        for (int n = 0; n < 4; ++n) {
            const T wn = (T)w[4 * m + n];
            q[n] = u0 * wn + q[n];
            q[4 + n] = u1 * wn + q[4 + n];
        }
    }
    for (int n = 0; n < 8; n += 2) {
        j[n] = fr * q[n] + (j[n] - fi * q[n + 1]);
        j[n + 1] = fr * q[n + 1] + (j[n + 1] + fi * q[n]);
    }
}

// XCD-aware block -> (item, tile): consecutive workgroup ids land on the 8
// XCDs round-robin.  On a large grid they stay in order: a few items are in
// flight at a time, each read by every XCD, and the XCDs get equal work whatever
// the items' sizes.  On a small one each XCD gets a contiguous range of items, so
// that the beam records of an item pass through one L2 (in order, a thousand
// workgroups would hold dozens of items).  In order, 11,000 to 59,000 beams in 2 to
// 256 orientations are 4 to 10 % slower in mixed precision and 0 to 6 % in FP64 on 12
// to 46 tiles (59,000 on 23: 1.11 and 1.06 ms); at 68, 91, 136 and 188 tiles neither
// order wins in most, and they lie within 4 % of each other (59,000 on 188: 7.21 and
// 7.25 ms; 5,870 near-forward beams on them, FP64, 1.54 and 1.61).
__device__ __forceinline__ bool map_block(int n_items, int n_tiles, int &item,
                                          int &tile)
{
    const int total = n_items * n_tiles;
    const int nblk = gridDim.x;
    const int per_xcd = (nblk + 7) / 8;
    const int bid = blockIdx.x;
    const int logical = n_tiles >= 64 ? bid : (bid % 8) * per_xcd + bid / 8;
    if (logical >= total)
        return false;
    item = logical / n_tiles;
    tile = logical - item * n_tiles;
    return true;
}

// ---------------------------------------------------------------------------
// Device work queue (work mode MBS_WORK_QUEUE).  plan_segments_kernel cuts
// every orientation into beam segments on the device (the host plan's rule:
// segments of max(min_segment, ceil(n_beams / want)) beams, at least one per
// orientation) and splits the (item, tile) units into 8 contiguous ranges,
// one per XCD, so the units of one item stay in one XCD's L2.  A persistent
// workgroup takes units from its XCD's range with an atomic counter and,
// when that range is empty, from the next XCDs' in turn; it exits when all
// eight are empty.  Each unit still writes its own partial sums, so results
// do not depend on which workgroup ran it.  With the eight counters in one line
// and every look at one an atomic addition, the 2,048 workgroups' last looks took
// 1 ms (24 orientations of 80-200 beams on 181 x 48 directions: 1.2 ms, now 0.12).
// ---------------------------------------------------------------------------
// The least beams of a segment, on the host and on the device.  A segment costs its
// workgroups a start and an end (tables, the first records, the sum's way out)
// worth some tens of beams, and its partial grid; a launch ends with workgroups
// idle for half a segment.  With N beams, T tiles and P workgroups at once the two
// are N T / (P seg) x cost and seg / 2: least at a multiple of sqrt(N T / P).
// With P = 1024 that is the multiple 4 for costs of some 30 beams.  The optimum is
// flat: kernel and reduction with 2.7 and with 6.4 against 4, over 1,900 to 136,000
// beams in 1 to 256 orientations on 12 to 203 tiles, take on the mean (least to most)
// mixed 1.01 (0.97 to 1.09) and 1.01 (0.96 to 1.09), FP64 1.01 (0.97 to 1.09) and 1.00
// (0.93 to 1.07), mixed on the vector ALU 1.00 (0.96 to 1.04) and 1.03 (0.97 to 1.09),
// the incoherent sum 1.04 (0.99 to 1.17) and 0.98 (0.85 to 1.02): one rule for all, and
// not the best for each.  At least four: 185 beams on 91 x 16 take 20 us with four or
// five, 23 with eight, 50 with 32.
__host__ __device__ inline int64_t min_segment(int64_t n_beams, int n_tiles)
{
    const int64_t seg = (int64_t)(sqrt((double)(n_beams * n_tiles)) / 8.0);
    return seg > 4 ? seg : 4;
}

struct QueueCursor {
    int range = -1;   // XCD range being drained (thread 0 only)
    int tried = 0;    // ranges found empty so far
};

__device__ __forceinline__ bool next_unit(int *__restrict__ queue, int n_tiles, QueueCursor &qc,
                                          int &s_unit, int &item, int &tile)
{
    if (threadIdx.x == 0) {
        if (qc.range < 0)
            qc.range = blockIdx.x & 7;
        int u = -1;
        while (qc.tried < 8) {
            int *next = queue + Q_NEXT + Q_LINE * qc.range;
            const int end = queue[Q_END + qc.range];
            // another XCD's range is looked at before its counter is changed: at
            // the end every workgroup passes all eight
            if (qc.tried == 0 || __hip_atomic_load(next, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT) < end) {
                const int t = atomicAdd(next, 1);
                if (t < end) {
                    u = t;
                    break;
                }
            }
            qc.range = (qc.range + 1) & 7;
            ++qc.tried;
        }
        s_unit = u;
    }
    __syncthreads();
    const int u = s_unit;
    __syncthreads();
    if (u < 0)
        return false;
    item = u / n_tiles;
    tile = u - item * n_tiles;
    return true;
}

// One workgroup: the segment plan of the resident batch, and the queue
// header.  ooff [n_orient + 1] device orientation offsets; want: the target
// item count; items has room for want + n_orient items (the plan never
// needs more: sum over o of ceil(n_o / seg) <= n_beams / seg + n_orient).
__global__ void __launch_bounds__(1024) plan_segments_kernel(
    const int64_t *__restrict__ ooff, int n_orient, int want, int n_tiles,
    WorkItem *__restrict__ items, int *__restrict__ queue)
{
    __shared__ int s_scan[1024];
    __shared__ int s_base;
    const int64_t nb = ooff[n_orient];
    const int64_t seg =
        max(min_segment(nb, n_tiles), (nb + (int64_t)want - 1) / max((int64_t)want, (int64_t)1));
    if (threadIdx.x == 0)
        s_base = 0;
    __syncthreads();
    for (int o0 = 0; o0 < n_orient; o0 += blockDim.x) {
        const int o = o0 + threadIdx.x;
        int64_t b0 = 0, n = 0;
        int kseg = 0;
        if (o < n_orient) {
            b0 = ooff[o];
            n = ooff[o + 1] - b0;
            kseg = (int)max((int64_t)1, (n + seg - 1) / seg);
        }
        // inclusive scan of the segment counts over this chunk
        s_scan[threadIdx.x] = kseg;
        __syncthreads();
        for (int off = 1; off < (int)blockDim.x; off <<= 1) {
            const int v = threadIdx.x >= (unsigned)off ? s_scan[threadIdx.x - off] : 0;
            __syncthreads();
            s_scan[threadIdx.x] += v;
            __syncthreads();
        }
        const int first = s_base + s_scan[threadIdx.x] - kseg;
        for (int i = 0; i < kseg; ++i)
            items[first + i] = WorkItem{o, o + 1, b0 + n * i / kseg, b0 + n * (i + 1) / kseg};
        __syncthreads();
        if (threadIdx.x == blockDim.x - 1)
            s_base += s_scan[threadIdx.x];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const int total = s_base;
        const int64_t units = (int64_t)total * n_tiles;
        queue[Q_ITEMS] = total;
        for (int x = 0; x < 8; ++x) {
            queue[Q_NEXT + Q_LINE * x] = (int)(units * x / 8);
            queue[Q_END + x] = (int)(units * (x + 1) / 8);
        }
    }
}

struct KernelArgs {
    const WorkItem *items;
    int n_items, n_tiles, cells, n_az;
    const double *tab;       // grid tables [DT_COUNT][cells]
    const double *hdr;       // [n_beams][HDR_STRIDE]
    const uint32_t *wb;      // [n_beams][WB_STRIDE]
    const double *ebeam;     // [n_beams][EB_STRIDE]
    const double *w64;       // [n_beams][W64_STRIDE]
    const PhasorNode *phasor;  // [kPhasorN] phasor nodes of the mixed kernels
    const double2 *turns;    // [kTabN] phasors of the FP64 kernels
    const double *vtx;       // [n_vert][VTX_STRIDE]
    const double *vx;        // [n_vert][VX_STRIDE]
    const int64_t *ooff;     // [n_orient+1]
    const double *weights;   // [n_orient]
    double k, eps1;
    double *out;             // Mueller mode: [n_items][cells][16]; Jones: [n_items][cells][8]
    double *out_ns;          // same shape, no-shadow (NS only)
    double *per_orient;      // [n_orient][cells][16] (PER only, Mueller mode)
    int *queue;              // work-queue header (queue mode), else null
    const float *tab32;      // FP32 u0, u1 [cells][DT32_COUNT] (mixed kernels)
    const int32_t *sidx;     // [n_beams] spectrum slot of each beam, -1: direct
    const float2 *fbuf;      // [spectrum beams][cells] F from the spectra
    int waves;               // MFMA kernel occupancy variant (0: the default)
};

// Mueller of one orientation's Jones sum, weighted, stored to (first) or
// added to (later orientations of the item) a lane-owned global cell: the
// running orientation sum lives in memory, not in registers -- it is touched
// once per orientation, against thousands of beams of work in between.
template <typename T>
__device__ __forceinline__ void flush_mueller(const T *j, double w, double *dst, bool first,
                                              double *per)
{
    double mm[16];
    for (int q = 0; q < 16; ++q)
        mm[q] = 0.0;
    add_mueller(mm, j, w);
    if (per)
        for (int q = 0; q < 16; ++q)
            per[q] = mm[q];
    if (first) {
        for (int q = 0; q < 16; ++q)
            dst[q] = mm[q];
    } else {
        for (int q = 0; q < 16; ++q)
            dst[q] += mm[q];
    }
}

// All pointers are separate __restrict__ kernel arguments: the per-orientation
// stores into `out` must be provably disjoint from the beam records for the
// compiler to keep reading those through the scalar cache.
//
// The sum is kept in the global frame, G[m][c] += F W[m][c] (24 accumulators, 48
// FMAs a beam with W in scalar registers), and turned into the Jones sum once per
// orientation or segment.  Rotating each beam (R = u . T, R Jp, F R Jp) took 56 and
// twelve LDS reads.  PREC 0: FP64; PREC 1, the mixed kernel on the vector ALU: FP32
// sums of W rounded to FP32 (137,000 beams on 541 x 96 directions: 21.2 ms,
// where each beam rotated, with its conversions, took 32 to 33).
template <int PREC, int NS, int JONES, int PER, int QUEUE>
__global__ __launch_bounds__(256) MBS_OCCUPANCY(PREC == 1 ? (NS || !JONES ? 6 : 7) : MBS_MIN_WAVES) void
diffract_kernel(
    const WorkItem *__restrict__ items, int n_items, int n_tiles, int cells, int n_az,
    const double *__restrict__ tab, const double *__restrict__ hdr,
    const double *__restrict__ w64, const double *__restrict__ vtx,
    const double *__restrict__ vx, const double *__restrict__ ebeam,
    const PhasorNode *__restrict__ phasor, const double2 *__restrict__ turns,
    const int64_t *__restrict__ ooff, const double *__restrict__ weights, double k, double eps1,
    double *__restrict__ out, double *__restrict__ out_ns, double *__restrict__ per_orient,
    int *__restrict__ queue, const float *__restrict__ tab32)
{
    using U = typename std::conditional<PREC == 1, float, double>::type;
    using U2 = typename std::conditional<PREC == 1, PhasorNode, double2>::type;
    // LDS: the phasor table (1024 entries of 16 bytes), and the sums over the
    // shadow beams of an orientation (NS), a column per lane
    constexpr int TN = PREC == 1 ? kPhasorN : kTabN;
    __shared__ U2 s_tab[TN];
    __shared__ U s_jx[NS ? 8 * 256 : 1];
    __shared__ int s_unit;
    int item = 0, tile = 0;
    if constexpr (!QUEUE) {
        if (!map_block(n_items, n_tiles, item, tile))
            return;
    }
    for (int i = threadIdx.x; i < TN; i += blockDim.x) {
        if constexpr (PREC == 1)
            s_tab[i] = phasor[i];
        else
            s_tab[i] = turns[i];
    }
    __syncthreads();
    QueueCursor qc;
    for (;;) {
    if constexpr (QUEUE) {
        if (!next_unit(queue, n_tiles, qc, s_unit, item, tile))
            return;
    }
    const int cell = tile * 256 + threadIdx.x;
    const bool live = cell < cells;
    const int c = live ? cell : cells - 1;  // dead lanes compute, never store
    double d[3];
    for (int q = 0; q < 3; ++q)
        d[q] = kPhasorN * tab[(size_t)(DT_DIR + q) * cells + c];
    // this lane's rotation vectors u0, u1 (6 each)
    const U *u;
    size_t ld;
    if constexpr (PREC == 1) {
        u = tab32 + (size_t)c * DT32_COUNT;
        ld = 1;
    } else {
        u = tab + (size_t)DT_U0 * cells + c;
        ld = cells;
    }
    const auto add_shadow = [&](const double *w, U fr, U fi) {
        U jx[8];
        for (int q = 0; q < 8; ++q)
            jx[q] = s_jx[q * 256 + threadIdx.x];
        rotate_add<U>(w, u, ld, fr, fi, jx);
        for (int q = 0; q < 8; ++q)
            s_jx[q * 256 + threadIdx.x] = jx[q];
    };
    const WorkItem it = items[item];
    for (int o = it.o_begin; o < it.o_end; ++o) {
        int64_t b0 = ooff[o], b1 = ooff[o + 1];
        if constexpr (JONES) {
            b0 = it.b_begin;
            b1 = it.b_end;
        }
        U sum[W64_STRIDE];  // G
        for (int q = 0; q < W64_STRIDE; ++q)
            sum[q] = 0;
        if constexpr (NS)
            for (int q = 0; q < 8; ++q)
                s_jx[q * 256 + threadIdx.x] = 0;
        const int nbeam = (int)(b1 - b0);  // 32-bit loop test (scalar unit)
        const double *eb = ebeam + (size_t)b0 * EB_STRIDE;
        const double *w = w64 + (size_t)b0 * W64_STRIDE;
        BeamRecord rec{};
        Lines ahead{};
        if (nbeam > 0)
            rec = load_record(eb);
        for (int ib = 0; ib < nbeam; ++ib, w += W64_STRIDE) {
            const double *h = hdr + (size_t)(b0 + ib) * HDR_STRIDE;
            const bool shadow = NS && (high_word(rec.v[EB_KIND]) & 1) != 0;
            if constexpr (PREC == 0) {
                double fr, fi;
                const uint64_t dead =
                    aperture_any_f64(rec.v, h, vtx, vx, d, s_tab, k, eps1, fr, fi);
                ahead.arrived();
                const bool counts = __builtin_amdgcn_inverse_ballot_w64(~dead);
                if (shadow) {
                    if (counts)
                        add_shadow(w, fr, fi);
                } else if (counts) {
                    add_rotated<double>(w, fr, fi, sum);
                }
                ahead.touch(w + (ib + 1 < nbeam ? W64_STRIDE : 0));
                eb += ib + 1 < nbeam ? EB_STRIDE : 0;
                rec = load_record(eb);
            } else {
                float fr, fs;
                aperture_mixed(rec.v, h, vtx, vx, d, s_tab, k, eps1, fr, fs);
                const float scale = low_float(rec.v[EB_SCALE]);
                ahead.arrived();
                fr *= scale;
                fs *= kSqrt2 * scale;
                if (shadow)
                    add_shadow(w, fr, fs);
                else
                    add_rotated<float>(w, fr, fs, sum);
                ahead.touch(w + (ib + 1 < nbeam ? W64_STRIDE : 0));
                eb += ib + 1 < nbeam ? EB_STRIDE : 0;
                rec = load_record(eb);
            }
        }
        U j[8] = {0, 0, 0, 0, 0, 0, 0, 0}, jn[8];
        add_jones<U>(sum, u, ld, j);
        if constexpr (NS)  // the sum without and with the shadow beams
            for (int q = 0; q < 8; ++q) {
                jn[q] = j[q];
                j[q] += s_jx[q * 256 + threadIdx.x];
            }
        if (!live)
            continue;
        if constexpr (JONES) {
            // Jones partials in the kernel's own precision (FP32 for the
            // mixed kernel: half the bytes, the same values)
            U *dst = reinterpret_cast<U *>(out) + ((size_t)item * cells + cell) * 8;
            for (int q = 0; q < 8; ++q)
                dst[q] = j[q];
            if constexpr (NS) {
                U *dn = reinterpret_cast<U *>(out_ns) + ((size_t)item * cells + cell) * 8;
                for (int q = 0; q < 8; ++q)
                    dn[q] = jn[q];
            }
        } else {
            const double w = weights[o];
            const bool first = (o == it.o_begin);
            double *per = PER ? per_orient + ((size_t)o * cells + abi_cell(cell, n_az, cells)) * 16
                              : nullptr;
            flush_mueller(j, w, out + ((size_t)item * cells + cell) * 16, first, per);
            if constexpr (NS)
                flush_mueller(jn, w, out_ns + ((size_t)item * cells + cell) * 16, first,
                              (double *)nullptr);
        }
    }
    if constexpr (!QUEUE)
        return;
    }
}

// Incoherent sum (MBS_INCOHERENT), FP64: per orientation the Mueller
// matrices of the single beams are added -- sum_b Mueller(d_b) rather than
// Mueller(sum_b d_b) -- so beams do not interfere.  Its M11 element, the sum
// of |d_b|^2 / 2, is what the reference's theta probe accumulates
// (theta_m11_kernel, src/cuda/GpuDiffraction.cu:1909-1957).  With d = F q, q = R Jp,
// the sixteen sums are those of |F|^2 q_i conj(q_j), of which the Mueller matrix is a
// linear function: 40 FMAs a beam where adding its elements took about 85.
// An item is a beam segment of one orientation, or a run of whole orientations (as
// in diffract_kernel's orientation mode); it writes its weighted sum, and
// reduce_mueller_kernel adds the items.  With whole orientations only, 16 of them
// on 181 x 48 directions kept half of the device busy, each beam waiting for the one
// before: 0.65 ms, now 0.30.
__global__ __launch_bounds__(256) MBS_OCCUPANCY(MBS_MIN_WAVES) void diffract_incoherent_kernel(
    const WorkItem *__restrict__ items, int n_items, int n_tiles, int cells,
    const double *__restrict__ tab, const double *__restrict__ hdr,
    const double *__restrict__ w64, const double *__restrict__ vtx,
    const double *__restrict__ vx, const double *__restrict__ ebeam,
    const double2 *__restrict__ turns, const int64_t *__restrict__ ooff,
    const double *__restrict__ weights, double k, double eps1, double *__restrict__ out)
{
    int item, tile;
    if (!map_block(n_items, n_tiles, item, tile))
        return;
    const int cell = tile * 256 + threadIdx.x;
    const bool live = cell < cells;
    const int c = live ? cell : cells - 1;  // dead lanes compute, never store
    double d[3], u[12];
    for (int q = 0; q < 3; ++q)
        d[q] = kPhasorN * tab[(size_t)(DT_DIR + q) * cells + c];
    __shared__ double2 s_tab[kTabN];
    for (int q = 0; q < 12; ++q)
        u[q] = tab[(size_t)(DT_U0 + q) * cells + c];
    for (int i = threadIdx.x; i < kTabN; i += blockDim.x)
        s_tab[i] = turns[i];
    __syncthreads();
    const WorkItem it = items[item];
    for (int o = it.o_begin; o < it.o_end; ++o) {
        double diag[4] = {0, 0, 0, 0}, re[6] = {0, 0, 0, 0, 0, 0}, im[6] = {0, 0, 0, 0, 0, 0};
        int64_t b0 = ooff[o], b1 = ooff[o + 1];
        if (it.b_end > it.b_begin) {  // a segment
            b0 = it.b_begin;
            b1 = it.b_end;
        }
        const int nbeam = (int)(b1 - b0);
        const double *eb = ebeam + (size_t)b0 * EB_STRIDE;
        const double *w = w64 + (size_t)b0 * W64_STRIDE;
        BeamRecord rec{};
        Lines ahead{};
        if (nbeam > 0)
            rec = load_record(eb);
        for (int ib = 0; ib < nbeam; ++ib, w += W64_STRIDE) {
            double fr, fi;
            const uint64_t dead =
                aperture_any_f64(rec.v, hdr + (size_t)(b0 + ib) * HDR_STRIDE, vtx, vx, d, s_tab,
                                 k, eps1, fr, fi);
            ahead.arrived();
            if (__builtin_amdgcn_inverse_ballot_w64(~dead)) {
                double q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < 6; ++e)  // q += u[e] W[e]
                    for (int n = 0; n < 4; ++n) {
                        q[n] = __builtin_fma(u[e], w[4 * e + n], q[n]);
                        q[4 + n] = __builtin_fma(u[6 + e], w[4 * e + n], q[4 + n]);
                    }
                const double p = __builtin_fma(fr, fr, fi * fi);
                double s[8];
                for (int e = 0; e < 8; ++e)
                    s[e] = p * q[e];
                int n = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double ir = s[2 * i], ii = s[2 * i + 1];
                    diag[i] = __builtin_fma(ir, q[2 * i], __builtin_fma(ii, q[2 * i + 1], diag[i]));
                    for (int j = i + 1; j < 4; ++j, ++n) {
                        const double jr = q[2 * j], ji = q[2 * j + 1];
                        re[n] = __builtin_fma(ir, jr, __builtin_fma(ii, ji, re[n]));
                        im[n] = __builtin_fma(ii, jr, __builtin_fma(-ir, ji, im[n]));
                    }
                }
            }
            ahead.touch(w + (ib + 1 < nbeam ? W64_STRIDE : 0));
            eb += ib + 1 < nbeam ? EB_STRIDE : 0;
            rec = load_record(eb);
        }
        if (!live)
            continue;
        // as add_mueller; pairs in the order 01 02 03 12 13 23
        double m[16];
        m[0] = 0.5 * ((diag[0] + diag[2]) + (diag[1] + diag[3]));
        m[1] = 0.5 * ((diag[0] + diag[2]) - (diag[1] + diag[3]));
        m[4] = 0.5 * ((diag[0] - diag[2]) + (diag[1] - diag[3]));
        m[5] = 0.5 * ((diag[0] - diag[2]) - (diag[1] - diag[3]));
        m[2] = -re[0] - re[5];
        m[3] = -im[5] - im[0];
        m[6] = re[5] - re[0];
        m[7] = im[5] - im[0];
        m[8] = -re[1] - re[4];
        m[9] = re[4] - re[1];
        m[12] = im[1] + im[4];
        m[13] = im[1] - im[4];
        m[10] = re[2] + re[3];
        m[11] = im[2] - im[3];
        m[14] = -im[2] - im[3];
        m[15] = re[2] - re[3];
        const double weight = weights[o];
        double *dst = out + ((size_t)item * cells + cell) * 16;
        const bool first = (o == it.o_begin);
        for (int q = 0; q < 16; ++q)
            dst[q] = (first ? 0.0 : dst[q]) + weight * m[q];
    }
}

// ---- coherent sum as a matrix contraction on MFMA (mixed precision) -------
//
// The rotation is linear in the beam's polarisation data: with the
// direction-only vectors u0, u1 (6 components each) and the per-beam complex
// W[m][c] = T0[m] Jp[0][c] + T1[m] Jp[1][c],
//   J[i][c](dir) = sum_b F_b(dir) (R_b Jp_b)[i][c]
//                = sum_m u_i[m](dir) G[m][c](dir),  G = sum_b F_b(dir) W_b[m][c].
// G is a complex [64 directions x beams] . [beams x 12] product per wave, a
// real one with two rows (Re F, Im F) per beam and N = 24 columns.
//
// It runs on v_mfma_f32_32x32x16_bf16 with both factors split into three BF16
// parts (x = h + m + l, 24 significant bits): the six products down to 2^-16
// relative, hh hm hl mh mm lh, are summed in FP32; the first one left out is
// ~2^-25.  The matrix cores run BF16 beside the vector ALU (64 FMAs plus two of
// these: 281 cycles a wave, against 257 for the FMAs alone), while the FP32
// form does not overlap with it at all on this device (64 FMAs plus two
// v_mfma_f32_32x32x2f32: 396 cycles), so the split costs its 12 vector
// instructions and saves 128 cycles a beam.
//
// One v_permlane32_swap gives lane l of both halves the two parts of direction
// l (block 0) and l + 32 (block 1): Re F in lanes 0-31, Im F in lanes 32-63, as
// K rows 0-7 and 8-15.  Each lane then holds 8 K entries in four words, (h, h)
// (m, m) (0, l) (0, h), against the record's words (h, m) (h, m) (0, h) (0, l).
typedef float f32x16 __attribute__((ext_vector_type(16)));
// Word 3 of a raw buffer resource on gfx9-family devices (32-bit data
// format; the element and index fields unused).
constexpr int kBufferRsrcWord3 = 0x00020000;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The A words of one value: its three BF16 parts by truncation (each exact:
// h + m + l == x), as (h, h) (m, m) (0, l) (0, h).  The remainders are FP32
// numbers whose top halves are the parts.
__device__ __forceinline__ bf16x8 split_words(uint32_t x)
{
    const uint32_t h = x & 0xffff0000u;
    const uint32_t r = __float_as_uint(__uint_as_float(x) - __uint_as_float(h));
    const uint32_t m = r & 0xffff0000u;
    const uint32_t l = __float_as_uint(__uint_as_float(r) - __uint_as_float(m));
    constexpr uint32_t kTops = 0x07060302;  // the top halves of both operands
    const u32x4 w = {__builtin_amdgcn_perm(x, x, kTops), __builtin_amdgcn_perm(r, r, kTops), l, h};
    return __builtin_bit_cast(bf16x8, w);
}

enum { G_LD = 25 };  // LDS row stride (floats) of the per-wave G transpose
static_assert(32 * G_LD >= 8 * 64, "the tile holds a wave's shadow sums");

// G (this wave's accumulators) -> this lane's Jones sum.  Accumulator v of
// lane l holds G[dir][n] with n = l % 32, dir = 8 (v/4) + 4 (l/32) + v % 4
// (+32 for the second block).  The two 32-direction blocks pass through one
// 32-row LDS tile in turn (half the LDS of staging both at once, which lets
// five workgroups share a CU).  Called by every thread of the block.
__device__ __forceinline__ void mfma_epilogue(const f32x16 &g0, const f32x16 &g1,
                                              float *__restrict__ sg,
                                              const float *__restrict__ u, int cells,
                                              float *j)
{
    const int lane = threadIdx.x & 63;
    const int n = lane & 31;
    for (int blk = 0; blk < 2; ++blk) {
        const f32x16 &g = blk ? g1 : g0;
        if (n < WB_COLS) {
            for (int v = 0; v < 16; ++v) {
                const int i = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                sg[i * G_LD + n] = g[v];
            }
        }
        __syncthreads();
        if ((lane >> 5) == blk) {
            const float *gr = sg + (lane & 31) * G_LD;
            for (int t = 0; t < 4; ++t) {  // t = 2 i + c
                const int i = t >> 1, c = t & 1;
                float re = 0.0f, im = 0.0f;
                for (int m = 0; m < 6; ++m) {
                    const float um = u[6 * i + m];
                    re = __builtin_fmaf(um, gr[4 * m + 2 * c], re);
                    im = __builtin_fmaf(um, gr[4 * m + 2 * c + 1], im);
                }
                j[2 * t] = re;
                j[2 * t + 1] = im;
            }
        }
        __syncthreads();
    }
}

// FSRC: beams with sidx[b] >= 0 take F from fbuf (the near-forward spectrum
// source) instead of the aperture integral.  WAVES: the occupancy the
// register allocation is held to (see MBS_MFMA_OCCUPANCY).
template <int NS, int JONES, int PER, int QUEUE, int FSRC = 0, int WAVES = MBS_MFMA_WAVES>
__global__ __launch_bounds__(256) MBS_MFMA_OCCUPANCY void diffract_mfma_kernel(
    const WorkItem *__restrict__ items, int n_items, int n_tiles, int cells, int n_az,
    const double *__restrict__ tab, const double *__restrict__ hdr,
    const double *__restrict__ w64, const uint32_t *__restrict__ wb,
    const double *__restrict__ vtx, const double *__restrict__ vx,
    const double *__restrict__ ebeam, const PhasorNode *__restrict__ phasor, const int64_t *__restrict__ ooff,
    const double *__restrict__ weights, double k, double eps1, double *__restrict__ out,
    double *__restrict__ out_ns, double *__restrict__ per_orient, int *__restrict__ queue,
    const float *__restrict__ tab32, const int32_t *__restrict__ sidx = nullptr,
    const float2 *__restrict__ fbuf = nullptr)
{
    __shared__ PhasorNode s_tab[kPhasorN];
    __shared__ float s_g[4 * 32 * G_LD];
    __shared__ int s_unit;
    int item = 0, tile = 0;
    if constexpr (!QUEUE) {
        if (!map_block(n_items, n_tiles, item, tile))
            return;
    }
    for (int i = threadIdx.x; i < kPhasorN; i += blockDim.x)
        s_tab[i] = phasor[i];
    QueueCursor qc;
    for (;;) {
    if constexpr (QUEUE) {
        if (!next_unit(queue, n_tiles, qc, s_unit, item, tile))
            return;
    }
    const int cell = tile * 256 + threadIdx.x;
    const bool live = cell < cells;
    const int c = live ? cell : cells - 1;  // dead lanes compute, never store
    double d[3];
    for (int q = 0; q < 3; ++q)
        d[q] = kPhasorN * tab[(size_t)(DT_DIR + q) * cells + c];
    // this lane's u0, u1, read by the epilogue straight from its 48-byte
    // FP32 record (once per work item; staging them in LDS cost 12 KB per
    // workgroup, and one base address keeps the loads from holding twelve)
    const float *u = tab32 + (size_t)c * DT32_COUNT;
    __syncthreads();  // the phasor table
    float *sg = s_g + (threadIdx.x >> 6) * 32 * G_LD;
    const int lane = threadIdx.x & 63;
    const WorkItem it = items[item];
    for (int o = it.o_begin; o < it.o_end; ++o) {
        int64_t b0 = ooff[o], b1 = ooff[o + 1];
        if constexpr (JONES) {
            b0 = it.b_begin;
            b1 = it.b_end;
        }
        f32x16 g0 = {}, g1 = {};
        // a 32-bit trip count: the scalar unit has no 64-bit ordered compare,
        // so a 64-bit loop test would go to the vector unit
        const int nbeam = (int)(b1 - b0);
        const double *eb = ebeam + (size_t)b0 * EB_STRIDE;
        // Re F', Im F' / sqrt(2) of beam b
        const auto field = [&](const BeamRecord &r, int64_t b, float &fr,
                               float &fs) __attribute__((always_inline)) {
            const double *h = hdr + (size_t)b * HDR_STRIDE;
            const int slot = FSRC ? __builtin_amdgcn_readfirstlane(sidx[b]) : -1;
            if (FSRC && slot >= 0) {
                const float2 f = fbuf[(size_t)slot * cells + c];
                const float inv = high_float(r.v[EB_SCALE]);
                fr = f.x * inv;
                fs = f.y * (kInvSqrt2 * inv);
            } else {
                aperture_mixed(r.v, h, vtx, vx, d, s_tab, k, eps1, fr, fs);
            }
        };
        // Shadow beams (one an orientation) are added on the vector ALU to a sum
        // of their own, kept in this wave's part of the epilogue's tile: out of
        // the no-shadow sum with one accumulator set, and near the forward peak,
        // where they are far the largest, out of the FP32 sum of the others.
        // They are looked for 64 at a time ahead of the loop below, which runs
        // over them too, with zeros for operands.  A branch in that loop held
        // scalars that then spilled to vector lanes, 9 vector instructions a beam
        // in a queue launch: 12.04 -> 11.10 ms (aggregate of 50 to 40,000 beams,
        // 541 x 96), 2.20 -> 2.14 (15,000 beams, two grids), 1.21 -> 1.16
        // (59,000 beams by orientation, 181 x 32)
        {
            float jx[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            for (int ib = 0; ib < nbeam; ib += 64) {
                bool ext = false;
                if (ib + lane < nbeam)
                    ext = high_word(eb[(size_t)(ib + lane) * EB_STRIDE + EB_KIND]) & 1;
                for (uint64_t left = __ballot(ext); left; left &= left - 1) {
                    const int64_t b = b0 + ib + __builtin_ctzll(left);
                    const BeamRecord r = load_record(ebeam + (size_t)b * EB_STRIDE);
                    float fr, fs;
                    field(r, b, fr, fs);
                    const float scale = low_float(r.v[EB_SCALE]);
                    rotate_add<float>(w64 + (size_t)b * W64_STRIDE, u, 1, fr * scale,
                                      fs * (kSqrt2 * scale), jx);
                }
            }
            for (int q = 0; q < 8; ++q)
                sg[64 * q + lane] = jx[q];
        }
        BeamRecord rec{};
        if (nbeam > 0)
            rec = load_record(eb);
        // this lane's B words: row lane / 32, column lane % 32; the columns
        // past 24 lie outside the record and read as zero
        const int col = lane & 31;
        const int lane_off = col < WB_COLS
                                 ? ((lane >> 5) * WB_COLS + col) * WB_WORDS * (int)sizeof(uint32_t)
                                 : WB_STRIDE * (int)sizeof(uint32_t);
        const uint32_t *w = wb + (size_t)b0 * WB_STRIDE;
        for (int ib = 0; ib < nbeam; ++ib) {
            const int64_t b = b0 + ib;
            // With the spectrum's pointers as well, the scalar registers are short:
            // a size made anew for each beam keeps the descriptor, which the
            // compiler would take as a whole, from spilling to vector lanes (eight
            // instructions a beam; 11,000 near-forward beams 1.53 ms, now 1.46)
            constexpr int kBytes = WB_STRIDE * (int)sizeof(uint32_t);
            int size = kBytes;
            if constexpr (FSRC)
                asm volatile("s_movk_i32 %0, %1" : "=s"(size) : "n"(kBytes));
            const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint32_t *>(w), 0, size, kBufferRsrcWord3);
            w += WB_STRIDE;
            const u32x4 bw = __builtin_amdgcn_raw_buffer_load_b128(wres, lane_off, 0, 0);
            float fr, fs;
            field(rec, b, fr, fs);
            // the next beam's record: after this one's last table read (LDS
            // reads and scalar loads share one wait counter), so that it
            // arrives while the contraction issues
            eb += ib + 1 < nbeam ? EB_STRIDE : 0;
            rec = load_record(eb);
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(fr),
                                                             __float_as_uint(fs), false, false);
            const bf16x8 bop = __builtin_bit_cast(bf16x8, bw);
            g0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(split_words(sw[0]), bop, g0, 0, 0, 0);
            g1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(split_words(sw[1]), bop, g1, 0, 0, 0);
        }
        float j[8], jn[8], jx[8];
        for (int q = 0; q < 8; ++q)
            jx[q] = sg[64 * q + lane];
        mfma_epilogue(g0, g1, sg, u, cells, j);
        for (int q = 0; q < 8; ++q) {
            jn[q] = j[q];
            j[q] += jx[q];
        }
        if (!live)
            continue;
        if constexpr (JONES) {
            // FP32 Jones partials (the sums are FP32)
            float *dst = reinterpret_cast<float *>(out) + ((size_t)item * cells + cell) * 8;
            for (int q = 0; q < 8; ++q)
                dst[q] = j[q];
            if constexpr (NS) {
                float *dn = reinterpret_cast<float *>(out_ns) + ((size_t)item * cells + cell) * 8;
                for (int q = 0; q < 8; ++q)
                    dn[q] = jn[q];
            }
        } else {
            const double w = weights[o];
            const bool first = (o == it.o_begin);
            double *per = PER ? per_orient + ((size_t)o * cells + abi_cell(cell, n_az, cells)) * 16
                              : nullptr;
            flush_mueller(j, w, out + ((size_t)item * cells + cell) * 16, first, per);
            if constexpr (NS)
                flush_mueller(jn, w, out_ns + ((size_t)item * cells + cell) * 16, first,
                              (double *)nullptr);
        }
    }
    if constexpr (!QUEUE)
        return;
    __syncthreads();  // the next unit overwrites s_g
    }
}

// Zero fill (used instead of a memset so that no memset node is ever recorded
// into a captured graph).
__global__ void zero_kernel(double *__restrict__ p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0.0;
}

// Sum of per-item Mueller partials in item order: res[c] = sum_i part[i][c].
__global__ void reduce_mueller_kernel(const double *__restrict__ part, int n_items,
                                      int cells, int n_az, double *__restrict__ res)
{
    // (Mueller-mode items are always planned on the host)
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)cells * 16;
    if (idx >= n)
        return;
    double s = 0.0;
    for (int i = 0; i < n_items; ++i)
        s += part[(size_t)i * n + idx];
    res[abi_cell((int)(idx / 16), n_az, cells) * 16 + idx % 16] = s;
}

// Jones segments -> Mueller: items are ordered by orientation; for each
// orientation the segment Jones sums are added in segment order, converted
// and accumulated with the orientation weight (TracerPOTotal.cpp:5985-5994).
//
// Its floor is the partials' bytes (read once; per-orientation grids written
// once).  A thread that walks a cell's items alone waits for one load after the
// other with too few threads in flight, so a workgroup takes 32 cells and SLICES
// equal slices of the item list.  Of an orientation that a slice's ends cut, the
// slices leave their parts in LDS and the slice where it ends adds them in order;
// the slices' Mueller sums are added in order too, so the result is reproducible.
// 1,988 items (256 orientations) on 181 x 32 directions with their grids kept: 1.42
// -> 0.18 ms (559 MB: 3.2 TB/s); 333 items on 541 x 96: 0.19 -> 0.11 ms (5.0 TB/s).
// blockIdx.y selects the full or the no-shadow grid.
enum { J2M_CELLS = 32 };

// The end of the run of items of orientation o that starts at i (< end).
__device__ __forceinline__ int orientation_end(const WorkItem *__restrict__ items, int i, int end,
                                               int o)
{
    // the next 32 items, one a lane of this half of the wave
    const int at = i + (threadIdx.x & 31);
    const uint64_t same =
        __builtin_amdgcn_ballot_w64(at < end && items[min(at, end - 1)].o_begin == o);
    const uint32_t half = (uint32_t)(same >> (threadIdx.x & 32));
    if (half != 0xffffffffu)
        return i + __builtin_ctz(~half);
    int lo = i + 31, hi = end;  // items[lo] is of o, items[hi] is not
    while (hi - lo > 1) {
        const int mid = lo + (hi - lo) / 2;
        if (items[mid].o_begin == o)
            lo = mid;
        else
            hi = mid;
    }
    return hi;
}

// Adds the Jones partials of items [i, end) of a cell to j, in order, four
// items' loads at a time.
template <typename T>
__device__ __forceinline__ void add_partials(const T *__restrict__ part, size_t stride, int i,
                                             int end, double *j)
{
    struct alignas(16) Jones {
        T v[8];
    };
    const T *src = part + (size_t)i * stride;
    for (; i + 4 <= end; i += 4, src += 4 * stride) {
        Jones p[4];
        for (int u = 0; u < 4; ++u)
            p[u] = *reinterpret_cast<const Jones *>(src + u * stride);
        for (int u = 0; u < 4; ++u)
            for (int q = 0; q < 8; ++q)
                j[q] += p[u].v[q];
    }
    for (; i < end; ++i, src += stride) {
        const Jones p = *reinterpret_cast<const Jones *>(src);
        for (int q = 0; q < 8; ++q)
            j[q] += p.v[q];
    }
}

template <typename T, int SLICES>
__global__ void __launch_bounds__(J2M_CELLS * SLICES)
    jones_to_mueller_kernel(const T *__restrict__ part, const T *__restrict__ part_ns,
                            const WorkItem *__restrict__ items, int n_items, int cells,
                            int n_az, const double *__restrict__ weights,
                            double *__restrict__ res, double *__restrict__ res_ns,
                            double *__restrict__ per_orient, const int *__restrict__ queue)
{
    __shared__ double s_head[SLICES][8][J2M_CELLS], s_tail[SLICES][8][J2M_CELLS];
    __shared__ int s_state[SLICES];
    if (queue)  // planned on the device
        n_items = queue[Q_ITEMS];
    if (blockIdx.y) {
        part = part_ns;
        res = res_ns;
        per_orient = nullptr;
    }
    const int l = threadIdx.x % J2M_CELLS, slice = threadIdx.x / J2M_CELLS;
    const int first = blockIdx.x * J2M_CELLS;
    const int cell = min(first + l, cells - 1);  // spare lanes compute, never store
    const bool live = first + l < cells;
    const size_t stride = (size_t)cells * 8;
    const T *src = part + (size_t)cell * 8;
    double m[16];
    for (int q = 0; q < 16; ++q)
        m[q] = 0.0;
    const auto convert = [&](const double *j, int o) {
        if (per_orient) {
            double po[16];
            for (int q = 0; q < 16; ++q)
                po[q] = 0.0;
            add_mueller(po, j, weights[o]);
            double *dst = per_orient + ((size_t)o * cells + abi_cell(cell, n_az, cells)) * 16;
            for (int q = 0; q < 16; ++q) {
                if (live)
                    dst[q] = po[q];
                m[q] += po[q];
            }
        } else {
            add_mueller(m, j, weights[o]);
        }
    };
    // this slice's items, and what it leaves: NONE, the first part of an
    // orientation (TAIL), or nothing but a middle part of one (MIDDLE; also an
    // empty slice, whose part is zero)
    enum { NONE, TAIL, MIDDLE };
    const int lo = (int)((int64_t)n_items * slice / SLICES);
    const int hi = (int)((int64_t)n_items * (slice + 1) / SLICES);
    int state = lo < hi ? NONE : MIDDLE;
    int ends = -1;  // the orientation from before that ends here
    if (lo == hi)
        for (int q = 0; q < 8; ++q)
            s_head[slice][q][l] = 0.0;
    for (int i = lo; i < hi;) {
        const int o = items[i].o_begin;
        const int to = orientation_end(items, i, n_items, o);
        const bool before = i == lo && i > 0 && items[i - 1].o_begin == o;
        double j[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        add_partials(src, stride, i, min(to, hi), j);
        if (before) {
            for (int q = 0; q < 8; ++q)
                s_head[slice][q][l] = j[q];
            if (to <= hi)
                ends = o;
            else
                state = MIDDLE;
        } else if (to > hi) {
            for (int q = 0; q < 8; ++q)
                s_tail[slice][q][l] = j[q];
            state = TAIL;
        } else {
            convert(j, o);
        }
        i = to;
    }
    if (l == 0)
        s_state[slice] = state;
    __syncthreads();
    if (ends >= 0) {
        int from = slice - 1;
        while (s_state[from] == MIDDLE)
            --from;
        double j[8];
        for (int q = 0; q < 8; ++q)
            j[q] = s_tail[from][q][l];
        for (int e = from + 1; e <= slice; ++e)
            for (int q = 0; q < 8; ++q)
                j[q] += s_head[e][q][l];
        convert(j, ends);
    }
    for (int h = 0; h < 2; ++h) {  // eight elements at a time
        __syncthreads();
        for (int q = 0; q < 8; ++q)
            s_head[slice][q][l] = m[8 * h + q];
        __syncthreads();
        for (int i = threadIdx.x; i < 8 * J2M_CELLS; i += J2M_CELLS * SLICES) {
            const int q = i % 8, at = i / 8;
            double sum = 0.0;
            for (int e = 0; e < SLICES; ++e)
                sum += s_head[e][q][at];
            if (first + at < cells)
                res[abi_cell(first + at, n_az, cells) * 16 + 8 * h + q] = sum;
        }
    }
}

// Azimuth (laboratory-alpha) average of an orientation-summed Mueller grid,
// one row per zenith: HandlerPOTotal::WriteMatricesToFile
// (src/handler/HandlerPOTotal.cpp:23-122).  Row t = [theta in degrees,
// 2 pi dcos, M11..M44] with Mbar = (1/nAz) sum_p M(p,t) L(-phi_p), where
// L(a) rotates the Stokes Q/U block by 2a (at the poles the plain mean is
// taken); then the pole forms of PoleMueller (src/handler/PoleMueller.h:25-55)
// and the solid-angle weight of ScatteringRange::Compute2PiDcos
// (src/handler/Handler.h:70-125) in the stable sin*sin form.  One wave per
// row; the 64 lanes stride over azimuths and combine by a fixed butterfly, so
// the result is deterministic.
// blockIdx.y selects one of several grids stored back to back (the
// per-orientation grids of an MBS_PER_ORIENT run).
__global__ void __launch_bounds__(64) azimuth_average_kernel(
    const double *__restrict__ m, const double *__restrict__ theta, int n_az, int n_zen,
    double az_step, double *__restrict__ rows)
{
    const int t = blockIdx.x;
    const int nZ = n_zen + 1;
    m += (size_t)blockIdx.y * n_az * nZ * 16;
    rows += (size_t)blockIdx.y * nZ * 18;
    const double th = theta[t];
    const double tol = 256.0 * 2.220446049250313e-16;
    const bool fwd = __builtin_fabs(th) <= tol;
    const bool bwd = __builtin_fabs(th - kPi) <= tol;
    double s[16];
    for (int q = 0; q < 16; ++q)
        s[q] = 0.0;
    for (int p = threadIdx.x; p < n_az; p += 64) {
        const double *c = m + ((size_t)p * nZ + t) * 16;
        double sn, cs;
        sincos(2.0 * (-(double)p * az_step), &sn, &cs);
        for (int r = 0; r < 4; ++r) {
            const double *row = c + 4 * r;
            if (fwd || bwd) {
                for (int q = 0; q < 4; ++q)
                    s[4 * r + q] += row[q];
            } else {
                s[4 * r + 0] += row[0];
                s[4 * r + 1] += row[1] * cs - row[2] * sn;
                s[4 * r + 2] += row[1] * sn + row[2] * cs;
                s[4 * r + 3] += row[3];
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1)
        for (int q = 0; q < 16; ++q)
            s[q] += __shfl_xor(s[q], off, 64);
    if (threadIdx.x != 0)
        return;
    for (int q = 0; q < 16; ++q)
        s[q] /= (double)n_az;
    if (fwd || bwd) {
        const double m00 = s[0], m33 = s[15], m03 = s[3];
        const double m11 = fwd ? 0.5 * (s[5] + s[10]) : 0.5 * (s[5] - s[10]);
        for (int q = 0; q < 16; ++q)
            s[q] = 0.0;
        s[0] = m00;
        s[5] = m11;
        s[10] = fwd ? m11 : -m11;
        s[15] = m33;
        s[3] = m03;
        s[12] = m03;
    }
    double lo, hi;
    if (t == 0) {
        lo = theta[0];
        hi = 0.5 * (theta[0] + theta[n_zen > 0 ? 1 : 0]);
    } else if (t == n_zen) {
        lo = 0.5 * (theta[n_zen - 1] + theta[n_zen]);
        hi = theta[n_zen];
    } else {
        lo = 0.5 * (theta[t - 1] + theta[t]);
        hi = 0.5 * (theta[t] + theta[t + 1]);
    }
    double *o = rows + (size_t)t * 18;
    o[0] = (th * 180.0) / kPi;  // RadToDeg, src/common/common.cpp:140-143
    o[1] = 2.0 * sin(0.5 * (lo + hi)) * sin(0.5 * (hi - lo)) * (2.0 * kPi);
    for (int q = 0; q < 16; ++q)
        o[2 + q] = s[q];
}

}  // namespace mbs
