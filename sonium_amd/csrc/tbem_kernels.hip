// Dense Burton–Miller assembly on gfx950 (FP64).
//
// Four kernels fill the N x N row-major complex matrix of
// build_tbem_system_with_beta_parallel (crates/sonium-bem/src/core/assembly/
// tbem.rs:1284-1466) for one wavenumber:
//
//   far_kernel   every off-diagonal pair with the 13-point rule on the whole
//                field panel (the unsubdivided leaf of generate_subelements,
//                regular.rs:124-321).  One lane per field panel (column),
//                rows streamed through the workgroup: the lane keeps its
//                panel in registers, the collocation point and normal are
//                uniform (scalar loads), and 64 lanes store 1 KiB of a row.
//                This is the FP64-VALU-bound kernel: 13 kernel evaluations
//                per pair, each about 40 FP64 instructions (far_sums).
//   near_kernel  overwrites the near pairs (level-0 ratio < 3) with the sum
//                over their subdivision leaves; one lane per leaf.
//   self_kernel  overwrites the diagonal: Stokes edge integral of the
//                hypersingular kernel plus Duffy-collapsed Gauss–Legendre on
//                the 3 x nsec2 sub-triangles (singular.rs:297-578), the
//                QuadratureParams::for_ka tier (singular.rs:51-85) chosen per
//                panel from k*size, and the free terms (tbem.rs:1330-1358).
//   bc_rhs_kernel  only when some field panel carries a nonzero BC value:
//                the sum over such columns of tbem.rs:1419-1435.
//
// plane_wave_kernel adds the incident-field right-hand side
// (incident.rs:807-834 with bem_solver.rs:5005-5034).

#include <cmath>
#include <type_traits>

#include "internal.hpp"

namespace sbh {
namespace {

constexpr double FOUR_PI = 12.566370614359172;  // 4.0 * PI, exact product

// TR13 (gauss.rs:526-540); weights are used times 0.5 (gauss.rs:117-130).
__constant__ double kTrS[13] = {0.333333333333333, 0.260345966079040, 0.260345966079040,
                                0.479308067841920, 0.065130102902216, 0.065130102902216,
                                0.869739794195568, 0.638444188569810, 0.048690315425316,
                                0.638444188569810, 0.312865496004874, 0.048690315425316,
                                0.312865496004874};
__constant__ double kTrT[13] = {0.333333333333333, 0.260345966079040, 0.479308067841920,
                                0.260345966079040, 0.065130102902216, 0.869739794195568,
                                0.065130102902216, 0.048690315425316, 0.638444188569810,
                                0.312865496004874, 0.638444188569810, 0.312865496004874,
                                0.048690315425316};
__constant__ double kTrW[13] = {-0.149570044467682, 0.175615257433208, 0.175615257433208,
                                0.175615257433208, 0.053347235608838, 0.053347235608838,
                                0.053347235608838, 0.077113760890257, 0.077113760890257,
                                0.077113760890257, 0.077113760890257, 0.077113760890257,
                                0.077113760890257};

// Local vertex and mid-side coordinates (singular.rs:119-124 CSI6/ETA6).
__constant__ double kCsi6[6] = {0.0, 1.0, 0.0, 0.5, 0.5, 0.0};
__constant__ double kEta6[6] = {0.0, 0.0, 1.0, 0.0, 0.5, 0.5};

// Gauss–Legendre nodes/weights for orders 1..8 (row = order), uploaded once
// per device from the host restatement of gauss.rs:14-103.
__constant__ double kGlX[9][8];
__constant__ double kGlW[9][8];

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }

// a * b + c with the uniform addend c read from an SGPR pair.  Written with
// __builtin_fma the compiler copies each Horner constant into a VGPR pair
// before the FMA; the three-address form with an SGPR source saves those
// moves and registers (the far kernel runs about 12% faster on 20480 panels).
// Pure arithmetic: no memory operand, so nothing is left in flight.
__device__ __forceinline__ double fma_vvs(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
}

// sin and cos of r for |r| <= pi/2: sin r = r + r^3 P(r^2) and
// cos r = 1 - r^2/2 + r^4 Q(r^2) with P, Q of degree 7 interpolating at
// Chebyshev nodes in r^2 (gen_sincos_coefficients.py; error below 3.6e-17 for
// sin and 1.6e-17 for cos).
__device__ __forceinline__ void sincos_half_period(double r, double* sp, double* cp) {
    const double r2 = r * r;
    constexpr double P0 = -0.16666666666666666, P1 = 0.008333333333333316, P2 = -0.00019841269841254974,
                     P3 = 2.7557319219163234e-06, P4 = -2.5052107616996182e-08, P5 = 1.6058977312464087e-10,
                     P6 = -7.643970296798572e-13, P7 = 2.7314447669863995e-15;
    constexpr double Q0 = 0.041666666666666664, Q1 = -0.001388888888888888, Q2 = 2.480158730157985e-05,
                     Q3 = -2.7557319221569563e-07, Q4 = 2.0876756602875463e-09, Q5 = -1.1470712272749466e-11,
                     Q6 = 4.7778779252458453e-14, Q7 = -1.5218638369243573e-16;
    double ps = __builtin_fma(r2, P7, P6);
    ps = fma_vvs(r2, ps, P5);
    ps = fma_vvs(r2, ps, P4);
    ps = fma_vvs(r2, ps, P3);
    ps = fma_vvs(r2, ps, P2);
    ps = fma_vvs(r2, ps, P1);
    ps = fma_vvs(r2, ps, P0);
    *sp = __builtin_fma(r * r2, ps, r);
    double pc = __builtin_fma(r2, Q7, Q6);
    pc = fma_vvs(r2, pc, Q5);
    pc = fma_vvs(r2, pc, Q4);
    pc = fma_vvs(r2, pc, Q3);
    pc = fma_vvs(r2, pc, Q2);
    pc = fma_vvs(r2, pc, Q1);
    pc = fma_vvs(r2, pc, Q0);
    *cp = __builtin_fma(r2 * r2, pc, __builtin_fma(-0.5, r2, 1.0));
}

// The same for |r| <= 0.32 (PANEL_PHASE_MAX) with P of degree 4 and Q of
// degree 3 ("panel" coefficients; error below 3e-19 for sin and 2e-17 for cos).
__device__ __forceinline__ void sincos_panel(double r, double* sp, double* cp) {
    const double r2 = r * r;
    constexpr double SP0 = -0.16666666666666666, SP1 = 0.00833333333333161, SP2 = -0.0001984126982781413,
                     SP3 = 2.7557282426861207e-06, SP4 = -2.501102979241046e-08;
    constexpr double SQ0 = 0.041666666666664874, SQ1 = -0.001388888888329103, SQ2 = 2.4801559965701305e-05,
                     SQ3 = -2.751459668586056e-07;
    double ps = __builtin_fma(r2, SP4, SP3);
    ps = fma_vvs(r2, ps, SP2);
    ps = fma_vvs(r2, ps, SP1);
    ps = fma_vvs(r2, ps, SP0);
    *sp = __builtin_fma(r * r2, ps, r);
    double pc = __builtin_fma(r2, SQ3, SQ2);
    pc = fma_vvs(r2, pc, SQ1);
    pc = fma_vvs(r2, pc, SQ0);
    pc = __builtin_fma(r2, pc, -0.5);
    *cp = __builtin_fma(r2, pc, 1.0);
}

// sin and cos of x for |x| < 2^20.  Cody & Waite (1980) two-constant
// reduction by pi with FMA, x = q pi + r, |r| <= pi/2, and both signs
// flipped for odd q.
__device__ __forceinline__ void sincos_red(double x, double* sp, double* cp) {
    constexpr double ONE_OVER_PI = 0.3183098861837907;
    constexpr double PI_HI = 3.141592653589793;
    constexpr double PI_LO = 1.2246467991473532e-16;
    const double q = __builtin_rint(x * ONE_OVER_PI);
    double r = __builtin_fma(-q, PI_HI, x);
    r = __builtin_fma(-q, PI_LO, r);
    double sr, cr;
    sincos_half_period(r, &sr, &cr);
    // (-1)^q: bit 0 of q moved to the sign bit of both results
    const unsigned long long sign = (unsigned long long)((unsigned)(int)q & 1u) << 63;
    *sp = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, sr) ^ sign);
    *cp = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, cr) ^ sign);
}
// 1/sqrt(d2) to about 1 ulp: the hardware estimate (24 correct bits) and one
// third-order (Householder) step, y1 = y0 (1 + e/2 + 3e^2/8) with
// e = 1 - d2 y0^2, whose truncation error (5/16) e^3 is below 1e-22.
__device__ __forceinline__ double rsqrt_nr(double d2) {
    const double y = __builtin_amdgcn_rsq(d2);
    const double e = __builtin_fma(-d2 * y, y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

struct Acc {
    double2 g, h, ht, e;
};

__device__ __forceinline__ Acc acc_zero() {
    Acc a;
    a.g = a.h = a.ht = a.e = make_double2(0.0, 0.0);
    return a;
}

// tbem.rs:1404-1417: matrix coefficient of a field panel for its BC.
__device__ __forceinline__ double2 coefficient(const Acc& r, const PanelBc& bc, double2 gamma,
                                               double2 tau, double2 beta, double2 iwr) {
    double2 c = make_double2(0.0, 0.0);
    if (bc.type == 0) {
        c = cadd(cmul(cmul(r.h, gamma), tau), cmul(r.e, beta));
    } else if (bc.type == 1) {
        double2 t = cadd(cmul(cmul(r.g, gamma), tau), cmul(r.ht, beta));
        c = make_double2(-t.x, -t.y);
    }
    if (bc.type == 0 && bc.has_adm) {
        double2 t = cadd(cmul(cmul(r.g, gamma), tau), cmul(r.ht, beta));
        c = csub(c, cmul(cmul(t, make_double2(bc.adm[0], bc.adm[1])), iwr));
    }
    return c;
}

// tbem.rs:1419-1435: BC right-hand-side contribution of a field panel.
__device__ __forceinline__ double2 bc_contribution(const Acc& r, const PanelBc& bc, double2 gamma,
                                                   double2 tau, double2 beta, double2 iwr) {
    double2 v = make_double2(bc.value[0], bc.value[1]);
    if (bc.type == 0) return cmul(cmul(cadd(cmul(cmul(r.g, gamma), tau), cmul(r.ht, beta)), v), iwr);
    if (bc.type == 1) return cmul(cadd(cmul(cmul(r.h, gamma), tau), cmul(r.e, beta)), v);
    return make_double2(0.0, 0.0);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ void wave_sum_acc(Acc& a) {
    a.g.x = wave_sum(a.g.x); a.g.y = wave_sum(a.g.y);
    a.h.x = wave_sum(a.h.x); a.h.y = wave_sum(a.h.y);
    a.ht.x = wave_sum(a.ht.x); a.ht.y = wave_sum(a.ht.y);
    a.e.x = wave_sum(a.e.x); a.e.y = wave_sum(a.e.y);
}

template <int CTRL>
__device__ __forceinline__ double dpp_read(double v) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned long long)(unsigned)lo);
}

// Sum over the 16 lanes of a DPP row; every lane of the row gets a total.
__device__ __forceinline__ double row16_sum(double v) {
    v += dpp_read<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_read<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_read<0x141>(v);  // row_half_mirror: lane i <- 7 - i within each half row
    v += dpp_read<0x140>(v);  // row_mirror: lane i <- 15 - i
    return v;
}

// The same over the 16 lanes of each row.
__device__ __forceinline__ void row16_sum_acc(Acc& a) {
    a.g.x = row16_sum(a.g.x); a.g.y = row16_sum(a.g.y);
    a.h.x = row16_sum(a.h.x); a.h.y = row16_sum(a.h.y);
    a.ht.x = row16_sum(a.ht.x); a.ht.y = row16_sum(a.ht.y);
    a.e.x = row16_sum(a.e.x); a.e.y = row16_sum(a.e.y);
}

// ---------------------------------------------------------------------------
// One quadrature point of the regular kernel, regular.rs:214-281.  DERIV also
// accumulates the analytic wavenumber derivative of every channel into dr
// (regular.rs:229-278), from the same point, as the reference's shared
// quadrature loop does.  The point evaluation uses 1/r from rsqrt_nr and FMA
// contraction (the reference divides by r nine times); the quadrature rules,
// subdivisions and channel formulas are the reference's.  The surrounding
// code keeps the reference's operation order (no contraction).
#pragma clang fp contract(off)

template <bool DERIV>
__device__ inline void ref_point_t(const double pos[3], double wga, const double src[3],
                                   const double srcn[3], const double nf[3], double wavruim, double k2,
                                   double k, double hf, Acc& r, Acc& dr) {
#pragma clang fp contract(on)
    const double d0 = pos[0] - src[0], d1 = pos[1] - src[1], d2 = pos[2] - src[2];
    const double dsq = d0 * d0 + d1 * d1 + d2 * d2;
    if (!(dsq > 1e-30)) return;  // |d| <= 1e-15: normalize() returns 0, then `dis < 1e-15` skips
    const double inv = rsqrt_nr(dsq);
    const double dis = dsq * inv;
    const double u0 = d0 * inv, u1 = d1 * inv, u2 = d2 * inv;
    const double re1 = wavruim * dis;
    const double re2 = (wga * (1.0 / FOUR_PI)) * inv;
    double s, c;
    sincos_red(re1, &s, &c);
    const double2 zg = make_double2(c * re2, s * re2);
    const double2 z1 = make_double2(-inv, wavruim);
    const double2 zb = cmul(zg, z1);
    const double re1_h = u0 * nf[0] + u1 * nf[1] + u2 * nf[2];
    const double re2_h = -(u0 * srcn[0] + u1 * srcn[1] + u2 * srcn[2]);
    const double rq = re1_h * re2_h;
    const double nxny = srcn[0] * nf[0] + srcn[1] * nf[1] + srcn[2] * nf[2];
    const double inv2 = inv * inv;
    const double t3 = 3.0 * rq + nxny;
    const double2 zef = make_double2((3.0 * inv2 - k2) * rq + nxny * inv2, -wavruim * inv * t3);
    r.g = cadd(r.g, zg);
    r.h = cadd(r.h, cscale(zb, re1_h));
    r.ht = cadd(r.ht, cscale(zb, re2_h));
    r.e = cadd(r.e, cmul(zg, zef));
    if (DERIV) {
        const double2 dzg = cmul(zg, make_double2(0.0, hf * dis));
        const double2 dzb = cadd(cmul(dzg, z1), cmul(zg, make_double2(0.0, hf)));
        const double2 dzef = make_double2(-2.0 * k * rq, -hf * inv * t3);
        dr.g = cadd(dr.g, dzg);
        dr.h = cadd(dr.h, cscale(dzb, re1_h));
        dr.ht = cadd(dr.ht, cscale(dzb, re2_h));
        dr.e = cadd(dr.e, cadd(cmul(dzg, zef), cmul(zg, dzef)));
    }
}

// Shape-function position of local (s, t) (regular.rs:682-690).
__device__ inline void shape_pos(const double* c, double s, double t, double p[3]) {
    double N0 = 1.0 - s - t;
    p[0] = 0.0 + N0 * c[0] + s * c[3] + t * c[6];
    p[1] = 0.0 + N0 * c[1] + s * c[4] + t * c[7];
    p[2] = 0.0 + N0 * c[2] + s * c[5] + t * c[8];
}

// Vertices of the leaf with path `code` (midpoint arithmetic is exact).
__device__ inline void decode_leaf(uint64_t code, double xi[3], double et[3]) {
    xi[0] = 0.0; xi[1] = 1.0; xi[2] = 0.0;
    et[0] = 0.0; et[1] = 0.0; et[2] = 1.0;
    int depth = (int)(code >> LEAF_DEPTH_SHIFT);
    for (int l = 0; l < depth; ++l) {
        int ch = (int)((code >> (2 * l)) & 3u);
        double mx[3] = {(xi[0] + xi[1]) / 2.0, (xi[1] + xi[2]) / 2.0, (xi[2] + xi[0]) / 2.0};
        double me[3] = {(et[0] + et[1]) / 2.0, (et[1] + et[2]) / 2.0, (et[2] + et[0]) / 2.0};
        if (ch == 3) {
            xi[0] = mx[0]; xi[1] = mx[1]; xi[2] = mx[2];
            et[0] = me[0]; et[1] = me[1]; et[2] = me[2];
        } else {
            int cm = (ch + 2) % 3;
            double x0 = xi[ch], e0 = et[ch];
            xi[0] = x0; xi[1] = mx[ch]; xi[2] = mx[cm];
            et[0] = e0; et[1] = me[ch]; et[2] = me[cm];
        }
    }
}

// Point q of a subdivided leaf (regular.rs:164-196): affine map of the TR13
// point into the leaf, weight times |det|, then compute_parameters.
template <bool DERIV>
__device__ inline void near_point_t(const PanelGeom& G, uint64_t code, int q, const double src[3],
                                    const double srcn[3], double wavruim, double k2, double k, double hf, Acc& r,
                                    Acc& dr) {
    double xi[3], et[3];
    decode_leaf(code, xi, et);
    double cs = kTrS[q], ec = kTrT[q], wg = kTrW[q] * 0.5;
    double l0 = 1.0 - cs - ec;
    double xio = xi[0] * l0 + xi[1] * cs + xi[2] * ec;
    double eto = et[0] * l0 + et[1] * cs + et[2] * ec;
    double dx1 = xi[1] - xi[0], dy1 = et[1] - et[0];
    double dx2 = xi[2] - xi[0], dy2 = et[2] - et[0];
    double det = fabs(dx1 * dy2 - dx2 * dy1);
    double weih2 = wg * det;
    double pos[3];
    shape_pos(G.c, xio, eto, pos);
    ref_point_t<DERIV>(pos, weih2 * G.jac, src, srcn, G.nf, wavruim, k2, k, hf, r, dr);
}

__device__ inline void near_point(const PanelGeom& G, uint64_t code, int q, const double src[3],
                                  const double srcn[3], double wavruim, double k2, Acc& r) {
    near_point_t<false>(G, code, q, src, srcn, wavruim, k2, 0.0, 0.0, r, r);
}

// Full TR13 on the unsubdivided panel in reference order (bc_rhs_kernel).
template <bool DERIV>
__device__ inline void full_point_t(const PanelGeom& G, int q, const double src[3], const double srcn[3],
                                    double wavruim, double k2, double k, double hf, Acc& r, Acc& dr) {
    double pos[3];
    shape_pos(G.c, kTrS[q], kTrT[q], pos);
    ref_point_t<DERIV>(pos, (kTrW[q] * 0.5) * G.jac, src, srcn, G.nf, wavruim, k2, k, hf, r, dr);
}

__device__ inline void full_point(const PanelGeom& G, int q, const double src[3], const double srcn[3],
                                  double wavruim, double k2, Acc& r) {
    full_point_t<false>(G, q, src, srcn, wavruim, k2, 0.0, 0.0, r, r);
}

struct SelfTier {
    int ngpo1, ngausin, nsec1, nsec2;
};

// singular.rs:51-85 QuadratureParams::for_ka
__device__ inline SelfTier tier_for(double ka) {
    if (ka < 0.3) return {3, 4, 4, 2};
    if (ka < 1.0) return {4, 5, 6, 2};
    if (ka < 2.0) return {5, 6, 8, 3};
    return {6, 7, 10, 4};
}

__device__ inline int self_samples(const SelfTier& t) {
    return 3 * t.nsec1 * t.ngpo1 + 3 * t.nsec2 * t.ngausin * t.ngausin;
}

// Sample s of the self-panel rule (singular.rs:322-410 edge part, :412-578
// bulk part).  Edge samples add to E only; bulk samples to G, H, Ht and
// E += k^2 G (n_x . n_y).  The sub-triangle loop repeats the second
// sub-triangle for every isec >= 1, as the reference does.  DERIV also adds
// the wavenumber derivatives (singular.rs:380-386, 509-545) to dr.
template <bool DERIV>
__device__ inline void self_sample_t(const PanelGeom& G, const SelfTier& t, int s, const double src[3],
                                     const double srcn[3], double wavruim, double k2, double k, double hf, Acc& r,
                                     Acc& dr) {
    const double* c = G.c;
    const int per_edge = t.nsec1 * t.ngpo1;
    const int nedge = 3 * per_edge;
    if (s < nedge) {
        int ieg = s / per_edge;
        int rem = s - ieg * per_edge;
        int isec = rem / t.ngpo1;
        int ig = rem - isec * t.ngpo1;
        int ig1 = (ieg + 1) % 3;
        double dpoi[3];
        double leneg = 0.0;
        for (int i = 0; i < 3; ++i) {
            dpoi[i] = c[3 * ig1 + i] - c[3 * ieg + i];
            leneg += dpoi[i] * dpoi[i];
        }
        leneg = sqrt(leneg);
        double dpoo[3] = {dpoi[0] / leneg, dpoi[1] / leneg, dpoi[2] / leneg};
        double leneg_scaled = leneg / (2.0 * (double)t.nsec1);
        double delsec = 2.0 / (double)t.nsec1;
        double secmid = -1.0 - delsec / 2.0;
        for (int k = 0; k <= isec; ++k) secmid += delsec;
        double sga = secmid + kGlX[t.ngpo1][ig] / (double)t.nsec1;
        double wga = kGlW[t.ngpo1][ig] * leneg_scaled;
        double diff[3];
        for (int i = 0; i < 3; ++i) {
            double crd = c[3 * ieg + i] + dpoi[i] * (sga + 1.0) / 2.0;
            diff[i] = crd - src[i];
        }
        double dis = sqrt(diff[0] * diff[0] + diff[1] * diff[1] + diff[2] * diff[2]);
        if (!(dis > 1e-15)) return;
        double u[3] = {diff[0] / dis, diff[1] / dis, diff[2] / dis};
        double re1 = wavruim * dis;
        double re2 = FOUR_PI * dis;
        double sn, cs;
        sincos_red(re1, &sn, &cs);
        double2 zg = make_double2(cs / re2, sn / re2);
        double2 z1 = make_double2(-1.0 / dis, wavruim);
        double2 zgf = cmul(zg, z1);
        double2 zd0 = cscale(zgf, u[0]), zd1 = cscale(zgf, u[1]), zd2 = cscale(zgf, u[2]);
        double2 w0 = csub(cscale(zd1, dpoo[2]), cscale(zd2, dpoo[1]));
        double2 w1 = csub(cscale(zd2, dpoo[0]), cscale(zd0, dpoo[2]));
        double2 w2 = csub(cscale(zd0, dpoo[1]), cscale(zd1, dpoo[0]));
        double2 dot = cadd(cadd(cscale(w0, srcn[0]), cscale(w1, srcn[1])), cscale(w2, srcn[2]));
        r.e = cadd(r.e, cscale(dot, wga));
        if (DERIV) {
            double2 dzg = cmul(zg, make_double2(0.0, hf * dis));
            double2 zgd = cadd(cmul(dzg, z1), cmul(zg, make_double2(0.0, hf)));
            double2 e0 = cscale(zgd, u[0]), e1 = cscale(zgd, u[1]), e2 = cscale(zgd, u[2]);
            double2 v0 = csub(cscale(e1, dpoo[2]), cscale(e2, dpoo[1]));
            double2 v1 = csub(cscale(e2, dpoo[0]), cscale(e0, dpoo[2]));
            double2 v2 = csub(cscale(e0, dpoo[1]), cscale(e1, dpoo[0]));
            double2 dd = cadd(cadd(cscale(v0, srcn[0]), cscale(v1, srcn[1])), cscale(v2, srcn[2]));
            dr.e = cadd(dr.e, cscale(dd, wga));
        }
        return;
    }
    s -= nedge;
    const int ng2 = t.ngausin * t.ngausin;
    const int per_edge_b = t.nsec2 * ng2;
    int ieg = s / per_edge_b;
    int rem = s - ieg * per_edge_b;
    int isec = rem / ng2;
    int rem2 = rem - isec * ng2;
    int i = rem2 / t.ngausin;
    int j = rem2 - i * t.ngausin;
    int ig1 = (ieg + 1) % 3;
    int ig2 = ieg + 3;
    const double* CSI6 = kCsi6;
    const double* ETA6 = kEta6;
    double aresub = 1.0 / 24.0 / (double)t.nsec2;
    double ss0 = 1.0 / 3.0, ts0 = 1.0 / 3.0, ss1, ss2, ts1, ts2;
    if (isec == 0) {
        ss1 = CSI6[ieg]; ss2 = CSI6[ig2]; ts1 = ETA6[ieg]; ts2 = ETA6[ig2];
    } else {
        ss1 = CSI6[ig2]; ss2 = CSI6[ig1]; ts1 = ETA6[ig2]; ts2 = ETA6[ig1];
    }
    double wei = kGlW[t.ngausin][i] * kGlW[t.ngausin][j];
    double sga = kGlX[t.ngausin][i], tga = kGlX[t.ngausin][j];
    double sgg = 0.5 * (1.0 - sga) * ss0 + 0.25 * (1.0 + sga) * ((1.0 - tga) * ss1 + (1.0 + tga) * ss2);
    double tgg = 0.5 * (1.0 - sga) * ts0 + 0.25 * (1.0 + sga) * ((1.0 - tga) * ts1 + (1.0 + tga) * ts2);
    double pos[3];
    shape_pos(c, sgg, tgg, pos);
    double wga = wei * (1.0 + sga) * aresub * G.jac;
    double d0 = pos[0] - src[0], d1 = pos[1] - src[1], d2 = pos[2] - src[2];
    double dis = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
    if (!(dis > 1e-15)) return;
    double u0 = d0 / dis, u1 = d1 / dis, u2 = d2 / dis;
    double re1 = wavruim * dis;
    double re2 = wga / (FOUR_PI * dis);
    double sn, cs;
    sincos_red(re1, &sn, &cs);
    double2 zg = make_double2(cs * re2, sn * re2);
    double2 z1 = make_double2(-1.0 / dis, wavruim);
    double2 zb = cmul(zg, z1);
    double re1_h = u0 * G.nf[0] + u1 * G.nf[1] + u2 * G.nf[2];
    double re2_h = -(u0 * srcn[0] + u1 * srcn[1] + u2 * srcn[2]);
    r.g = cadd(r.g, zg);
    r.h = cadd(r.h, cscale(zb, re1_h));
    r.ht = cadd(r.ht, cscale(zb, re2_h));
    double nd = srcn[0] * G.nf[0] + srcn[1] * G.nf[1] + srcn[2] * G.nf[2];
    r.e = cadd(r.e, cscale(cscale(zg, k2), nd));
    if (DERIV) {
        double2 dzg = cmul(zg, make_double2(0.0, hf * dis));
        double2 dzb = cadd(cmul(dzg, z1), cmul(zg, make_double2(0.0, hf)));
        dr.g = cadd(dr.g, dzg);
        dr.h = cadd(dr.h, cscale(dzb, re1_h));
        dr.ht = cadd(dr.ht, cscale(dzb, re2_h));
        dr.e = cadd(dr.e, cscale(cadd(cscale(dzg, k2), cscale(zg, 2.0 * k)), nd));
    }
}

__device__ inline void self_sample(const PanelGeom& G, const SelfTier& t, int s, const double src[3],
                                   const double srcn[3], double wavruim, double k2, Acc& r) {
    self_sample_t<false>(G, t, s, src, srcn, wavruim, k2, 0.0, 0.0, r, r);
}

// Parameters of a derivative assembly d/dp (tbem.rs:1858-2019): dk/dp = ws,
// beta and its total derivative, i rho omega and its derivative, and
// dY/dp = adm_scale * Y.
struct DerivParams {
    double k, wavruim, hf, tau_r, sign, ws, adm_scale;
    double2 beta, beta_d, iwr, iwr_d;
};

// d_cb and d_hb of one pair (tbem.rs:1972-1977); b = values, d = derivatives.
__device__ inline void deriv_blocks(const Acc& b, const Acc& d, const DerivParams& P, double2* d_cb, double2* d_hb) {
    const double2 gamma = make_double2(1.0, 0.0);
    const double2 tau = make_double2(P.tau_r, 0.0);
    *d_cb = cadd(cadd(cscale(cmul(cmul(d.h, gamma), tau), P.ws), cscale(cmul(d.e, P.beta), P.ws)),
                 cmul(b.e, P.beta_d));
    *d_hb = cadd(cadd(cscale(cmul(cmul(d.g, gamma), tau), P.ws), cscale(cmul(d.ht, P.beta), P.ws)),
                 cmul(b.ht, P.beta_d));
}

__device__ inline double2 h_block(const Acc& b, const DerivParams& P) {
    return cadd(cmul(cmul(b.g, make_double2(1.0, 0.0)), make_double2(P.tau_r, 0.0)), cmul(b.ht, P.beta));
}

// Matrix derivative of one pair for the field panel's BC (tbem.rs:1978-1995).
__device__ inline double2 deriv_from_blocks(double2 d_cb, double2 d_hb, double2 h_b, const PanelBc& bc,
                                            const DerivParams& P) {
    if (bc.type == 0) {
        double2 v = cscale(d_cb, P.sign);
        if (bc.has_adm) {
            const double2 y = make_double2(bc.adm[0], bc.adm[1]);
            v = csub(v, cmul(cscale(y, P.sign), cadd(cmul(d_hb, P.iwr), cmul(h_b, P.iwr_d))));
            v = csub(v, cmul(cmul(cscale(cscale(y, P.adm_scale), P.sign), h_b), P.iwr));
        }
        return v;
    }
    if (bc.type == 1) return cscale(d_hb, -P.sign);
    return make_double2(0.0, 0.0);
}

__device__ inline double2 deriv_coefficient(const Acc& b, const Acc& d, const PanelBc& bc, const DerivParams& P) {
    double2 d_cb, d_hb;
    deriv_blocks(b, d, P, &d_cb, &d_hb);
    return deriv_from_blocks(d_cb, d_hb, h_block(b, P), bc, P);
}

// Right-hand-side derivative of a nonzero-BC field panel (tbem.rs:1998-2013).
__device__ inline double2 deriv_bc_contribution(const Acc& b, const Acc& d, const PanelBc& bc, const DerivParams& P) {
    double2 d_cb, d_hb;
    deriv_blocks(b, d, P, &d_cb, &d_hb);
    const double2 sv = cscale(make_double2(bc.value[0], bc.value[1]), P.sign);
    if (bc.type == 0) return cmul(sv, cadd(cmul(d_hb, P.iwr), cmul(h_block(b, P), P.iwr_d)));
    if (bc.type == 1) return cmul(sv, d_cb);
    return make_double2(0.0, 0.0);
}

// Source free terms of the derivative (tbem.rs:1896-1915).
__device__ inline void deriv_free_terms(const PanelBc& bc, const DerivParams& P, double2* diag, double2* rhs) {
    const double2 tau = make_double2(P.tau_r, 0.0);
    const double2 btd = cadd(cmul(P.iwr_d, P.beta), cmul(P.iwr, P.beta_d));
    double2 dg = make_double2(0.0, 0.0), rh = make_double2(0.0, 0.0);
    if (bc.type == 0) {
        if (bc.has_adm) {
            const double2 y = make_double2(bc.adm[0], bc.adm[1]);
            dg = csub(dg, cscale(cmul(cmul(cscale(y, P.sign), btd), tau), 0.5));
            const double2 yd = cscale(y, P.adm_scale);
            dg = csub(dg, cscale(cmul(cmul(cmul(cscale(yd, P.sign), P.iwr), P.beta), tau), 0.5));
        }
        const double2 avg = make_double2(bc.value[0], bc.value[1]);
        rh = cadd(rh, cscale(cmul(cmul(cscale(avg, P.sign), btd), tau), 0.5));
    } else if (bc.type == 1) {
        dg = cadd(dg, cscale(cmul(cscale(P.beta_d, P.sign), tau), 0.5));
    }
    *diag = dg;
    *rhs = rh;
}

#pragma clang fp contract(on)

// Per-panel constants of the TR13 points y_q = v0 + s_q e1 + t_q e2 of the
// frequency-family kernel: the Gram entries of the two edges.
struct FamilyPoints {
    double e11, e12x2, e22;  // e1.e1, 2 e1.e2, e2.e2
};

__device__ __forceinline__ FamilyPoints family_points(const FarPanel& P) {
    FamilyPoints f;
    f.e11 = P.e1[0] * P.e1[0] + P.e1[1] * P.e1[1] + P.e1[2] * P.e1[2];
    f.e12x2 = 2.0 * (P.e1[0] * P.e2[0] + P.e1[1] * P.e2[1] + P.e1[2] * P.e2[2]);
    f.e22 = P.e2[0] * P.e2[0] + P.e2[1] * P.e2[1] + P.e2[2] * P.e2[2];
    return f;
}

// 13-point sums of one (collocation point, field panel) pair: the matrix
// factors cb = H tau + E beta and, in MODE 1, hb = G tau + Ht beta
// (tbem.rs:1404-1417 with gamma = 1).
//
// What bounds it is the FP64 VALU issue rate: 13 evaluations per pair, each a
// square root, a sine and a cosine.  Everything that can be is moved out of
// the evaluation:
//  - Geometry from the panel centre.  With the corners at c + V_i (V_0 + V_1 +
//    V_2 = 0) the rule's points are c, c + kappa V_i (two groups of three) and
//    c + a V_i + b V_j + c V_k (the six permutations), so with A = |c - x|^2,
//    D_i = (c - x).V_i:  |y - x|^2 = A + 2 kappa D_i + kappa^2 |V_i|^2, two FMAs
//    (three in the group of six, whose |displacement|^2 is kept per panel),
//    and the projection on n_x takes one or two.
//  - Phase from the panel centre.  e^{ikr} = e^{ik r_c} e^{ik(r - r_c)}: the first
//    factor multiplies the finished sums, and the difference stays below
//    k times the panel radius, so sine and cosine need no reduction and, on
//    a resolved mesh, a short polynomial (sincos_panel).  The centre point's
//    own difference is zero.
//  - Lengths in units of 1/k (FAR_LONG, FAR_SHORT), so that k is one.
//  - One complex weight per point.  With y = 1/r, u = y^2, g = -(y_q - x).n_x,
//    pr = (y_q - x).n_y (constant on a flat panel), rq = pr g u and
//    t = 3 rq + n_x.n_y,
//      H = sum z pr y (-y + ik),  E = sum z [(t u - k^2 rq) - ik t y],
//      G = sum z,                 Ht = sum z g y (-y + ik),   z = w e^{ikr} y,
//    so tau and an imaginary beta (the Burton-Miller factor i/k) enter the real
//    and the imaginary part of one weight each, and cb takes four FMAs.
//  - The rule's four weights multiply the sums of their groups.
// Per evaluation this takes 41 FP64 instructions (529 a pair, pair work included)
// where separate channel sums over a reduced sine took 68; the assembly of 20480
// panels takes 8.0 ms instead of 13.2, of which this loop 7.8 instead of 12.0.
//
// Variants (far_variant): FAR_SHORT and FAR_LONG need a purely imaginary beta
// and a phase difference within the range of their polynomials; FAR_GENERAL
// takes any k and beta, with lengths as they are and a full reduction.
constexpr double TR_A = 0.048690315425316, TR_B = 0.312865496004874, TR_C = 0.638444188569810;
constexpr double TR_K1 = 0.479308067841920 - 0.260345966079040;  // first group of three: c + K1 V_i
constexpr double TR_K2 = 0.869739794195568 - 0.065130102902216;  // second group of three
constexpr double TR_W0 = -0.149570044467682, TR_W1 = 0.175615257433208, TR_W2 = 0.053347235608838,
                 TR_W3 = 0.077113760890257;

// Uniform values of a launch, in units of 1/s: s = k and kap = 1, or s = 1 and kap = k.
struct FarUniform {
    double s, kap, tau, br, bi;  // br + i bi = beta s
};

template <int VAR>
__device__ __forceinline__ FarUniform far_uniform(double k, double tau, double2 beta) {
    FarUniform u;
    u.s = VAR == FAR_GENERAL ? 1.0 : k;
    u.kap = VAR == FAR_GENERAL ? k : 1.0;
    u.tau = tau;
    u.br = beta.x * u.s;
    u.bi = beta.y * u.s;
    return u;
}

// A field panel as the far loop keeps it: corner 0 and centre offset (exact
// lengths), V_1, V_2 and the squares below in units of 1/s.
struct FarLane {
    double v0[3], cv[3], V1[3], V2[3], nf[3];
    double L[3];  // |V_i|^2
    double Q[6];  // |displacement|^2 of the group of six
    double wj;
};

__device__ __forceinline__ double dot3(const double* a, const double* b) {
    return __builtin_fma(a[2], b[2], __builtin_fma(a[1], b[1], a[0] * b[0]));
}

// The squares of a lane's corner offsets and of its group of six.
__device__ __forceinline__ void lane_squares(FarLane& f) {
    const double V0[3] = {-(f.V1[0] + f.V2[0]), -(f.V1[1] + f.V2[1]), -(f.V1[2] + f.V2[2])};
    f.L[0] = dot3(V0, V0);
    f.L[1] = dot3(f.V1, f.V1);
    f.L[2] = dot3(f.V2, f.V2);
    // |a V_i + b V_j + c V_k|^2 = (a-b)(a-c)|V_i|^2 + (b-a)(b-c)|V_j|^2 + (c-a)(c-b)|V_k|^2, all terms
    // with V_0 + V_1 + V_2 = 0
    constexpr double qa = (TR_A - TR_B) * (TR_A - TR_C), qb = (TR_B - TR_A) * (TR_B - TR_C),
                     qc = (TR_C - TR_A) * (TR_C - TR_B);
#pragma unroll
    for (int m = 0; m < 6; ++m) {
        const int i = m >> 1, j = (i + 1 + (m & 1)) % 3, k = 3 - i - j;  // a on corner i, b on j, c on k
        f.Q[m] = __builtin_fma(qa, f.L[i], __builtin_fma(qb, f.L[j], qc * f.L[k]));
    }
}

__device__ __forceinline__ FarLane far_lane(const FarPanel& P, double s) {
    FarLane f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        f.v0[d] = P.v0[d];
        f.cv[d] = (P.e1[d] + P.e2[d]) * (1.0 / 3.0);
        f.V1[d] = s * (P.e1[d] - f.cv[d]);
        f.V2[d] = s * (P.e2[d] - f.cv[d]);
        f.nf[d] = P.nf[d];
    }
    lane_squares(f);
    f.wj = P.wj;
    return f;
}

// Calls point(d2, g, centre, sums) for the 13 points and add(weight, sums) for
// each weight group.  Ap is A as the caller's ordering of the points left it.
template <typename Part, typename Point, typename Add>
__device__ __forceinline__ void far_points(const FarLane& P, double A, const double& Ap, const double* D, double gc,
                                           const double* g, const Part& zero, Point&& point, Add&& add) {
    {
        Part a = zero;
        point(A, gc, true, a);
        add(TR_W0, a);
    }
    {
        Part a = zero;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            point(__builtin_fma(TR_K1 * TR_K1, P.L[i], __builtin_fma(2.0 * TR_K1, D[i], Ap)),
                  __builtin_fma(TR_K1, g[i], gc), false, a);
        add(TR_W1, a);
    }
    {
        Part a = zero;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            point(__builtin_fma(TR_K2 * TR_K2, P.L[i], __builtin_fma(2.0 * TR_K2, D[i], Ap)),
                  __builtin_fma(TR_K2, g[i], gc), false, a);
        add(TR_W2, a);
    }
    {
        Part a = zero;
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            // displacement (a - c) V_i + (b - c) V_j, c the weight of the third corner
            const int i = m >> 1, j = (i + 1 + (m & 1)) % 3;
            constexpr double ac = TR_A - TR_C, bc = TR_B - TR_C;
            point(__builtin_fma(2.0 * ac, D[i], __builtin_fma(2.0 * bc, D[j], Ap + P.Q[m])),
                  __builtin_fma(ac, g[i], __builtin_fma(bc, g[j], gc)), false, a);
        }
        add(TR_W3, a);
    }
}

// sin and cos of a phase difference in the variant's range (VAR's k times length).
template <int VAR>
__device__ __forceinline__ void sincos_difference(double x, double* sn, double* cs) {
    if (VAR == FAR_GENERAL)
        sincos_red(x, sn, cs);
    else if (VAR == FAR_LONG)
        sincos_half_period(x, sn, cs);
    else
        sincos_panel(x, sn, cs);
}

template <int MODE, int VAR>
__device__ __forceinline__ void far_sums(const FarLane& P, const Source& src, const FarUniform& K, double2& cb,
                                         double2& hb) {
    double x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        x[d] = (P.v0[d] - src.c[d]) + P.cv[d];
        if (VAR != FAR_GENERAL) x[d] *= K.s;
    }
    const double A = dot3(x, x);
    const double D1 = dot3(x, P.V1), D2 = dot3(x, P.V2);
    const double pr = dot3(x, P.nf);
    const double nn = dot3(src.n, P.nf);
    // g of the centre and its slopes; MODE 0 carries g pr (times beta, imaginary) instead
    const double gm = MODE == 0 && VAR != FAR_GENERAL ? -K.bi * pr : VAR != FAR_GENERAL ? -K.bi : -1.0;
    const double gc = gm * dot3(x, src.n);
    const double g1 = gm * dot3(P.V1, src.n), g2 = gm * dot3(P.V2, src.n);
    const double D[3] = {-(D1 + D2), D1, D2};
    const double g[3] = {-(g1 + g2), g1, g2};
    const double P1 = K.tau * pr;
    const double N = VAR != FAR_GENERAL ? K.bi * nn : nn;
    const double kap2 = K.kap * K.kap;
    const double yc = rsqrt_nr(A);
    const double rc = VAR == FAR_GENERAL ? K.kap * (A * yc) : A * yc;
    struct Part {
        double cr, ci, hr, hi;
    };
    // Orders the points: the next one's distance waits for this one's sums.  Left to itself the compiler
    // interleaves all 13 (256 registers, one or two waves per SIMD).
    double Ap = A;
    auto after = [&](Part& a) {
        if (MODE == 0)
            asm volatile("" : "+v"(Ap), "+v"(a.cr), "+v"(a.ci));
        else
            asm volatile("" : "+v"(Ap), "+v"(a.cr), "+v"(a.ci), "+v"(a.hr), "+v"(a.hi));
    };
    // One point: distance d2, projection gq, added to a (phase difference zero at the centre).
    auto point = [&](double d2, double gq, bool centre, Part& a) {
        const double y = rsqrt_nr(d2);
        const double u = y * y;
        double sn = 0.0, cs = 1.0;
        if (!centre)
            sincos_difference<VAR>(VAR == FAR_GENERAL ? __builtin_fma(K.kap, d2 * y, -rc)
                                                      : __builtin_fma(d2, y, -rc), &sn, &cs);
        double wr, wi;
        if (VAR != FAR_GENERAL) {
            const double R = (MODE == 0 ? gq : pr * gq) * u;  // beta rq
            const double T = __builtin_fma(3.0, R, N);        // beta t
            wr = u * __builtin_fma(-P1, y, T);
            wi = __builtin_fma(y, __builtin_fma(T, u, -R), P1 * u);
        } else {
            const double rq = (pr * gq) * u;
            const double t = __builtin_fma(3.0, rq, nn);
            const double er = __builtin_fma(t, u, -kap2 * rq), ei = -K.kap * (t * y);
            wr = y * (__builtin_fma(K.br, er, -K.bi * ei) - P1 * u);
            wi = y * __builtin_fma(K.kap * P1, y, __builtin_fma(K.br, ei, K.bi * er));
        }
        a.cr = __builtin_fma(cs, wr, a.cr);
        a.ci = __builtin_fma(cs, wi, a.ci);
        if (!centre) {
            a.cr = __builtin_fma(-sn, wi, a.cr);
            a.ci = __builtin_fma(sn, wr, a.ci);
        }
        if (MODE == 1) {
            double vr, vi;
            if (VAR != FAR_GENERAL) {
                vr = __builtin_fma(-gq, u, K.tau * y);  // y (tau - beta g y), imaginary beta
                vi = -gq * (u * y);
            } else {
                const double hr = -u, hi = K.kap * y;  // y (-y + ik)
                vr = y * __builtin_fma(gq, __builtin_fma(K.br, hr, -K.bi * hi), K.tau);
                vi = y * (gq * __builtin_fma(K.br, hi, K.bi * hr));
            }
            a.hr = __builtin_fma(cs, vr, a.hr);
            a.hi = __builtin_fma(cs, vi, a.hi);
            if (!centre) {
                a.hr = __builtin_fma(-sn, vi, a.hr);
                a.hi = __builtin_fma(sn, vr, a.hi);
            }
        }
        after(a);
    };
    Part tot = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](double w, const Part& a) {
        tot.cr = __builtin_fma(w, a.cr, tot.cr);
        tot.ci = __builtin_fma(w, a.ci, tot.ci);
        if (MODE == 1) {
            tot.hr = __builtin_fma(w, a.hr, tot.hr);
            tot.hi = __builtin_fma(w, a.hi, tot.hi);
        }
    };
    far_points(P, A, Ap, D, gc, g, Part{0.0, 0.0, 0.0, 0.0}, point, add);
    double sn, cs;
    sincos_red(rc, &sn, &cs);
    const double fh = P.wj * K.s, fc = fh * K.s;
    cb = make_double2(fc * __builtin_fma(cs, tot.cr, -sn * tot.ci), fc * __builtin_fma(cs, tot.ci, sn * tot.cr));
    if (MODE == 1)
        hb = make_double2(fh * __builtin_fma(cs, tot.hr, -sn * tot.hi), fh * __builtin_fma(cs, tot.hi, sn * tot.hr));
}

// Matrix coefficient of a field panel from its two factors (tbem.rs:1404-1417).
__device__ __forceinline__ double2 column_coefficient(double2 cb, double2 hb, const PanelBc& bc, double2 iwr) {
    if (bc.type == 1) return make_double2(-hb.x, -hb.y);
    double2 c = make_double2(0.0, 0.0);
    if (bc.type == 0) {
        c = cb;
        if (bc.has_adm) c = csub(c, cmul(cmul(hb, make_double2(bc.adm[0], bc.adm[1])), iwr));
    }
    return c;
}

// Far entry of one pair.
template <int MODE, int VAR>
__device__ __forceinline__ double2 far_entry(const FarLane& P, const Source& S, const PanelBc& bc,
                                             const FarUniform& K, double2 iwr) {
    double2 cb, hb;
    far_sums<MODE, VAR>(P, S, K, cb, hb);
    return MODE == 0 ? cb : column_coefficient(cb, hb, bc, iwr);
}

// Rigid/vibrating coefficient (H * gamma) * tau + E * beta with gamma = 1.
__device__ __forceinline__ double2 velocity_coefficient(double hr, double hi, double er, double ei, double tau_r,
                                                        double2 beta) {
    return make_double2(hr * tau_r + (er * beta.x - ei * beta.y), hi * tau_r + (er * beta.y + ei * beta.x));
}

// ---------------------------------------------------------------------------
// Far kernel.  MODE 0: every field panel has a velocity BC without
// admittance (rigid or vibrating body), so only H and E are needed and
// A_ij = H*gamma*tau + E*beta.  MODE 1: general per-column coefficients.
//
// Row maxima for the low-precision copy (rowmax non-null, rows_per_block <=
// FAR_MAX_ROWS): the block also writes, per row i, the maximum of
// max(|Re A_ij|, |Im A_ij|) over its 256 columns at rowmax[i * nbx +
// blockIdx.x], leaving out the near pairs and the diagonal that the later
// kernels overwrite (they fold their entries into rowmax[i * nbx + nbx - 1]
// as bit patterns with an atomic max; the column-0 blocks clear that slot).
constexpr int FAR_MAX_ROWS = 16;

template <int MODE, int VAR>
__global__ __launch_bounds__(256) void far_kernel(const FarPanel* __restrict__ panels,
                                                  const Source* __restrict__ sources,
                                                  const PanelBc* __restrict__ bcs, int64_t n,
                                                  int64_t lda, int rows_per_block, double k,
                                                  double tau_r, double2 beta, double2 iwr,
                                                  double2* __restrict__ A, const int64_t* __restrict__ row_ptr,
                                                  const NearPair* __restrict__ pairs, double* __restrict__ rowmax,
                                                  int64_t nbx) {
    __shared__ double smax[FAR_MAX_ROWS][256];
    __shared__ unsigned nmask[FAR_MAX_ROWS][8];
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool active = j < n;
    const int64_t jj = active ? j : n - 1;
    const FarUniform K = far_uniform<VAR>(k, tau_r, beta);
    const FarLane P = far_lane(panels[jj], K.s);
    PanelBc bc;
    if (MODE == 1) bc = bcs[jj];
    const int64_t i0 = (int64_t)blockIdx.y * rows_per_block;
    const int64_t i1 = min(n, i0 + rows_per_block);
    const int64_t c0 = (int64_t)blockIdx.x * 256;
    // This block's rows own one contiguous range of the row-sorted near-pair
    // list.  Its first 512 pairs are loaded into registers here, so the loads
    // complete behind the row loop; the near mask is built after it.
    int64_t e0 = 0, e1 = 0;
    int near_r[2] = {-1, -1}, near_c[2] = {0, 0};
    if (rowmax) {
        if (threadIdx.x < FAR_MAX_ROWS * 8) nmask[threadIdx.x >> 3][threadIdx.x & 7] = 0u;
        e0 = row_ptr[i0];
        e1 = row_ptr[i1];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t e = e0 + threadIdx.x + 256 * u;
            if (e < e1) {
                near_r[u] = pairs[e].i - (int)i0;
                near_c[u] = (int)((int64_t)pairs[e].j - c0);
            }
        }
    }
    for (int64_t i = i0; i < i1; ++i) {
        const double2 out = far_entry<MODE, VAR>(P, sources[i], bc, K, iwr);
        if (active) A[i * lda + j] = out;
        if (rowmax) smax[i - i0][threadIdx.x] = active ? fmax(fabs(out.x), fabs(out.y)) : 0.0;
    }
    if (rowmax) {
        __syncthreads();  // the mask was cleared by every wave before its row loop
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (near_r[u] >= 0 && near_c[u] >= 0 && near_c[u] < 256)
                atomicOr(&nmask[near_r[u]][near_c[u] >> 5], 1u << (near_c[u] & 31));
        for (int64_t e = e0 + 512 + threadIdx.x; e < e1; e += 256) {
            const NearPair np = pairs[e];
            const int64_t c = (int64_t)np.j - c0;
            if (c >= 0 && c < 256) atomicOr(&nmask[np.i - i0][c >> 5], 1u << (c & 31));
        }
        __syncthreads();
        // per row: the maximum over the columns that are neither near pairs nor the diagonal
        const int r = threadIdx.x >> 4, seg = threadIdx.x & 15;
        double m = 0.0;
        if (i0 + r < i1) {
            const unsigned bits = nmask[r][seg >> 1] >> (16 * (seg & 1));
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const int col = seg * 16 + c;
                const bool skip = ((bits >> c) & 1u) != 0u || c0 + col == i0 + r;
                m = fmax(m, skip ? 0.0 : smax[r][col]);
            }
        }
        __syncthreads();
        smax[r][seg] = m;
        __syncthreads();
        if (threadIdx.x < FAR_MAX_ROWS && i0 + threadIdx.x < i1) {
            double mm = 0.0;
#pragma unroll
            for (int c = 0; c < 16; ++c) mm = fmax(mm, smax[threadIdx.x][c]);
            const int64_t i = i0 + threadIdx.x;
            rowmax[i * nbx + blockIdx.x] = mm;
            if (blockIdx.x == 0) rowmax[i * nbx + nbx - 1] = 0.0;
        }
    }
}

// Folds max(|Re v|, |Im v|) of a near or diagonal entry into the row's slot
// (non-negative doubles order like their bit patterns; NaN entries are
// skipped, as fmax skips them).
__device__ __forceinline__ void fold_row_max(double* slot, double2 v) {
    const double m = fmax(fabs(v.x), fabs(v.y));
    if (m == m) atomicMax(reinterpret_cast<unsigned long long*>(slot), (unsigned long long)__double_as_longlong(m));
}

// Near pairs.  A subdivision leaf is a triangle similar to its panel: centre c +
// offset and corners at +-2^-depth V_i from it (the centre child of a cell is
// turned around, and the labels of a cell's corners rotate, which a symmetric
// rule does not see).  Every leaf is at least three of its sizes away, so its 13
// points take the far loop's evaluation, and one lane takes one leaf.
// What bounded the former wave per pair was everything but the evaluation: each
// lane decoded the leaf of its point, interpolated a position, and eight channel
// sums crossed the wave; 577620 pairs with 4.71 million leaves (20480 panels)
// took 1.13 ms, and take 0.18.
__device__ __forceinline__ FarLane leaf_lane(const FarPanel& P, uint64_t code, double s) {
    const int depth = (int)(code >> LEAF_DEPTH_SHIFT);
    double w0 = 0.0, w1 = 0.0, w2 = 0.0, size = 1.0;
    int rot = 0;  // corner m of the cell points along V_{(m + rot) % 3}
    for (int l = 0; l < depth; ++l) {
        const int ch = (int)((code >> (2 * l)) & 3u);
        const int d = ch + rot >= 3 ? ch + rot - 3 : ch + rot;
        size *= 0.5;
        if (ch == 3) {
            size = -size;
            rot = rot == 0 ? 2 : rot - 1;
        } else {
            w0 += d == 0 ? size : 0.0;
            w1 += d == 1 ? size : 0.0;
            w2 += d == 2 ? size : 0.0;
            rot = d;
        }
    }
    FarLane f;
    const double a1 = w1 - w0, a2 = w2 - w0, ss = s * size;  // V_0 = -V_1 - V_2
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double cv = (P.e1[d] + P.e2[d]) * (1.0 / 3.0);
        const double V1 = P.e1[d] - cv, V2 = P.e2[d] - cv;
        f.v0[d] = P.v0[d];
        f.cv[d] = __builtin_fma(a1, V1, __builtin_fma(a2, V2, cv));
        f.V1[d] = ss * V1;
        f.V2[d] = ss * V2;
        f.nf[d] = P.nf[d];
    }
    lane_squares(f);
    f.wj = P.wj * (size * size);  // the leaf's share of the panel's area
    return f;
}

// Sums over the leaves of pairs [p0, p0 + np) (np <= 256), by the whole
// workgroup: lane per leaf, 256 leaves at a time; each pair's leaves are added
// in order by one thread, so the sum depends on the pair alone.
// eval(pair, code) gives a leaf's double2; put(t, pair, sum) takes pair p0 + t's sum
// on thread t.
template <typename Eval, typename Put>
__device__ __forceinline__ void near_pairs(const NearPair* __restrict__ pairs, int64_t p0, int np,
                                           const uint64_t* __restrict__ leaves, Eval&& eval, Put&& put) {
    __shared__ int off[257];
    __shared__ double2 res[256];
    const int t = threadIdx.x;
    const NearPair mine = pairs[p0 + min(t, np - 1)];
    __syncthreads();  // the previous call's sums have been taken
    off[t + 1] = t < np ? mine.count : 0;
    if (t == 0) off[0] = 0;
    for (int d = 1; d < 256; d <<= 1) {  // inclusive scan
        __syncthreads();
        const int v = t >= d ? off[t + 1 - d] : 0;
        __syncthreads();
        off[t + 1] += v;
    }
    __syncthreads();
    const int total = off[np];
    const int b = off[t], e = off[t + 1];
    double2 sum = make_double2(0.0, 0.0);
    for (int base = 0; base < total; base += 256) {
        const int l = base + t;
        if (l < total) {
            int lo = 0, hi = np - 1;  // the last pair whose leaves start at or before l
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (off[mid] <= l) lo = mid; else hi = mid - 1;
            }
            const NearPair np_l = pairs[p0 + lo];
            res[t] = eval(np_l, leaves[np_l.begin + (l - off[lo])]);
        }
        __syncthreads();
        for (int q = max(b, base); q < min(e, base + 256); ++q) sum = cadd(sum, res[q - base]);
        __syncthreads();
    }
    if (t < np) put(t, mine, sum);
}

// Diagonal entry and BC free-term right-hand side of panel G (self integral
// summed by one wave, tbem.rs:1330-1358); every lane returns the totals.
// G refers to global memory: the sample loop indexes its nodes by edge.
__device__ __forceinline__ void self_entry(const PanelGeom& G, const Source& src, const PanelBc& bc, double k,
                                           double wavruim, double tau_r, double2 beta, double2 iwr, int lane,
                                           double2* diag_out, double2* rhs_out) {
    const double k2 = k * k;
    const SelfTier t = tier_for(k * G.size);
    const int ns = self_samples(t);
    Acc a = acc_zero();
    for (int s = lane; s < ns; s += 64) self_sample(G, t, s, src.c, src.n, wavruim, k2, a);
    wave_sum_acc(a);
    const double2 gamma = make_double2(1.0, 0.0);
    const double2 tau = make_double2(tau_r, 0.0);
    double2 diag = make_double2(0.0, 0.0);
    double2 local_rhs = make_double2(0.0, 0.0);
    double2 avg = make_double2(bc.value[0], bc.value[1]);
    // tbem.rs:1344-1358
    if (bc.type == 0) {
        diag = csub(diag, cscale(gamma, 0.5));
        if (bc.has_adm) {
            double2 adm = make_double2(bc.adm[0], bc.adm[1]);
            diag = csub(diag, cscale(cmul(cmul(cmul(adm, iwr), beta), tau), 0.5));
        }
        local_rhs = cadd(local_rhs, cscale(cmul(cmul(cmul(avg, iwr), beta), tau), 0.5));
    } else if (bc.type == 1) {
        diag = cadd(diag, cscale(cmul(beta, tau), 0.5));
        local_rhs = csub(local_rhs, cscale(cmul(avg, gamma), 0.5));
    }
    *diag_out = cadd(diag, coefficient(a, bc, gamma, tau, beta, iwr));
    *rhs_out = local_rhs;
}

__device__ __forceinline__ PanelBc rigid_bc() {
    PanelBc bc;
    bc.type = 0;
    bc.has_adm = 0;
    bc.value[0] = bc.value[1] = 0.0;
    bc.adm[0] = bc.adm[1] = 0.0;
    return bc;
}

// pairs_per_block near pairs per workgroup.
template <int MODE, int VAR>
__global__ __launch_bounds__(256) void near_kernel(const NearPair* __restrict__ pairs, int64_t npairs,
                                                   int pairs_per_block, const uint64_t* __restrict__ leaves,
                                                   const FarPanel* __restrict__ panels,
                                                   const Source* __restrict__ sources,
                                                   const PanelBc* __restrict__ bcs, int64_t lda, double k,
                                                   double tau_r, double2 beta, double2 iwr,
                                                   double2* __restrict__ A, double* __restrict__ rowmax,
                                                   int64_t nbx) {
    const int64_t p0 = (int64_t)blockIdx.x * pairs_per_block;
    const FarUniform K = far_uniform<VAR>(k, tau_r, beta);
    near_pairs(
        pairs, p0, (int)min((int64_t)pairs_per_block, npairs - p0), leaves,
        [&](const NearPair& np, uint64_t code) {
            PanelBc bc;
            if (MODE == 1) bc = bcs[np.j];
            return far_entry<MODE, VAR>(leaf_lane(panels[np.j], code, K.s), sources[np.i], bc, K, iwr);
        },
        [&](int, const NearPair& np, double2 v) {
            A[(int64_t)np.i * lda + np.j] = v;
            if (rowmax) fold_row_max(rowmax + (int64_t)np.i * nbx + nbx - 1, v);
        });
}

// One wave per panel: self integrals, free terms, BC free-term RHS.
__global__ __launch_bounds__(256) void self_kernel(const PanelGeom* __restrict__ geom,
                                                   const Source* __restrict__ sources,
                                                   const PanelBc* __restrict__ bcs, int general,
                                                   int64_t n, int64_t lda, double k, double wavruim,
                                                   double tau_r, double2 beta, double2 iwr,
                                                   double2* __restrict__ A, double2* __restrict__ rhs,
                                                   double* __restrict__ rowmax, int64_t nbx) {
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    const PanelBc bc = general ? bcs[i] : rigid_bc();
    double2 diag, local_rhs;
    self_entry(geom[i], sources[i], bc, k, wavruim, tau_r, beta, iwr, lane, &diag, &local_rhs);
    if (lane == 0) {
        A[i * lda + i] = diag;
        rhs[i] = local_rhs;
        if (rowmax) fold_row_max(rowmax + i * nbx + nbx - 1, diag);
    }
}

// ---------------------------------------------------------------------------
// Parameter derivative of the stabilized system (tbem.rs:1858-2019 and the
// CUDA workspace's assemble_wavenumber_derivative, tbem.rs:4399-4591): the same
// routes and launch structure as the value assembly, each pair producing its
// values b and wavenumber derivatives d from one pass over its points.

// Far sums with derivatives (harmonic factor +1), in the form of far_sums: one
// complex weight per point for each of the factors that a column needs.  With
// z = w e^{ikr} y, r = 1/y, dG/dk = i r G and d/dk[G (ik - 1/r)] = -k r G:
//   dH  = -k pr sum z              dE  = sum z [k (rq + n_x.n_y) - i k^2 r rq]
//   dG  = i sum z r                dHt = -k sum z g
// (in dE the i t/r terms of dz ef and z def cancel), so with p = dk/dp and the
// derivative beta' of beta
//   d_cb = p (dH tau + dE beta) + E beta',  d_hb = p (dG tau + dHt beta) + Ht beta',
//   hb   = G tau + Ht beta                  (tbem.rs:1972-1977).
// MODE 0 (velocity panels without admittance) needs d_cb only.  The variants
// are those of far_sums, chosen on the real parts of both beta and beta'.
struct DerivUniform {
    double s, kap, tau, wt;    // wt = p tau
    double br, bi;             // beta s
    double pbr, pbi, dbr, dbi; // p beta s and beta' s^2
};

template <int VAR>
__device__ __forceinline__ DerivUniform deriv_uniform(const DerivParams& P) {
    DerivUniform u;
    u.s = VAR == FAR_GENERAL ? 1.0 : P.k;
    u.kap = VAR == FAR_GENERAL ? P.k : 1.0;
    u.tau = P.tau_r;
    u.wt = P.ws * P.tau_r;
    u.br = P.beta.x * u.s;
    u.bi = P.beta.y * u.s;
    u.pbr = P.ws * u.br;
    u.pbi = P.ws * u.bi;
    u.dbr = P.beta_d.x * (u.s * u.s);
    u.dbi = P.beta_d.y * (u.s * u.s);
    return u;
}

template <int MODE, int VAR>
__device__ __forceinline__ void far_sums_d(const FarLane& P, const Source& src, const DerivUniform& K, double2& d_cb,
                                           double2& d_hb, double2& hb) {
    double x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        x[d] = (P.v0[d] - src.c[d]) + P.cv[d];
        if (VAR != FAR_GENERAL) x[d] *= K.s;
    }
    const double A = dot3(x, x);
    const double D1 = dot3(x, P.V1), D2 = dot3(x, P.V2);
    const double pr = dot3(x, P.nf);
    const double nn = dot3(src.n, P.nf);
    const double gm = MODE == 0 ? -pr : -1.0;  // MODE 0 carries g pr
    const double gc = gm * dot3(x, src.n);
    const double g1 = gm * dot3(P.V1, src.n), g2 = gm * dot3(P.V2, src.n);
    const double D[3] = {-(D1 + D2), D1, D2};
    const double g[3] = {-(g1 + g2), g1, g2};
    const double kap2 = K.kap * K.kap;
    const double yc = rsqrt_nr(A);
    const double rc = A * yc;
    const double c0 = -K.wt * K.kap * pr, bn = K.pbi * nn;
    struct Part {
        double cr, ci, hr, hi, vr, vi;
    };
    double Ap = A;
    auto after = [&](Part& a) {  // one point at a time, as in far_sums
        if (MODE == 0)
            asm volatile("" : "+v"(Ap), "+v"(a.cr), "+v"(a.ci));
        else
            asm volatile("" : "+v"(Ap), "+v"(a.cr), "+v"(a.ci), "+v"(a.hr), "+v"(a.hi), "+v"(a.vr), "+v"(a.vi));
    };
    auto point = [&](double d2, double gq, bool centre, Part& a) {
        const double y = rsqrt_nr(d2);
        const double u = y * y;
        const double r = d2 * y;
        double sn = 0.0, cs = 1.0;
        if (!centre) sincos_difference<VAR>(VAR == FAR_GENERAL ? K.kap * (r - rc) : r - rc, &sn, &cs);
        const double rq = (MODE == 0 ? gq : pr * gq) * u;
        const double t = __builtin_fma(3.0, rq, nn);
        double wr, wi;
        if (VAR != FAR_GENERAL) {
            wr = y * __builtin_fma(K.dbi, t * y, __builtin_fma(K.pbi * r, rq, c0));
            wi = y * __builtin_fma(K.dbi, __builtin_fma(t, u, -rq), __builtin_fma(K.pbi, rq, bn));
        } else {
            const double X = K.kap * (rq + nn), Z = -kap2 * (r * rq);
            const double F = __builtin_fma(t, u, -kap2 * rq), H = -K.kap * (t * y);
            wr = y * (c0 + __builtin_fma(K.pbr, X, -K.pbi * Z) + __builtin_fma(K.dbr, F, -K.dbi * H));
            wi = y * (__builtin_fma(K.pbr, Z, K.pbi * X) + __builtin_fma(K.dbr, H, K.dbi * F));
        }
        auto put = [&](double vr, double vi, double& ar, double& ai) {
            ar = __builtin_fma(cs, vr, ar);
            ai = __builtin_fma(cs, vi, ai);
            if (!centre) {
                ar = __builtin_fma(-sn, vi, ar);
                ai = __builtin_fma(sn, vr, ai);
            }
        };
        put(wr, wi, a.cr, a.ci);
        if (MODE == 1) {
            if (VAR != FAR_GENERAL) {
                const double gu = gq * u;  // g y times the y of z
                put(-K.dbi * gu, y * __builtin_fma(-K.dbi, gu, __builtin_fma(-K.pbi, gq, K.wt * r)), a.hr, a.hi);
                put(__builtin_fma(-K.bi, gu, K.tau * y), -K.bi * (gu * y), a.vr, a.vi);
            } else {
                const double kg = K.kap * gq, gy = gq * y;
                put(y * (gy * __builtin_fma(-K.dbr, y, -K.dbi * K.kap) - K.pbr * kg),
                    y * (__builtin_fma(K.wt, r, -K.pbi * kg) + gy * __builtin_fma(K.dbr, K.kap, -K.dbi * y)), a.hr,
                    a.hi);
                put(y * __builtin_fma(gy, __builtin_fma(-K.br, y, -K.bi * K.kap), K.tau),
                    y * (gy * __builtin_fma(K.br, K.kap, -K.bi * y)), a.vr, a.vi);
            }
        }
        after(a);
    };
    Part tot = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto add = [&](double w, const Part& a) {
        tot.cr = __builtin_fma(w, a.cr, tot.cr);
        tot.ci = __builtin_fma(w, a.ci, tot.ci);
        if (MODE == 1) {
            tot.hr = __builtin_fma(w, a.hr, tot.hr);
            tot.hi = __builtin_fma(w, a.hi, tot.hi);
            tot.vr = __builtin_fma(w, a.vr, tot.vr);
            tot.vi = __builtin_fma(w, a.vi, tot.vi);
        }
    };
    far_points(P, A, Ap, D, gc, g, Part{0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, point, add);
    double sn, cs;
    sincos_red(K.kap * rc, &sn, &cs);
    const double f0 = P.wj, f1 = P.wj * K.s;
    d_cb = make_double2(f1 * __builtin_fma(cs, tot.cr, -sn * tot.ci), f1 * __builtin_fma(cs, tot.ci, sn * tot.cr));
    if (MODE == 1) {
        d_hb = make_double2(f0 * __builtin_fma(cs, tot.hr, -sn * tot.hi), f0 * __builtin_fma(cs, tot.hi, sn * tot.hr));
        hb = make_double2(f1 * __builtin_fma(cs, tot.vr, -sn * tot.vi), f1 * __builtin_fma(cs, tot.vi, sn * tot.vr));
    }
}

template <int MODE, int VAR>
__global__ __launch_bounds__(256) void far_deriv_kernel(const FarPanel* __restrict__ panels,
                                                        const Source* __restrict__ sources,
                                                        const PanelBc* __restrict__ bcs, int64_t n, int64_t lda,
                                                        int rows_per_block, DerivParams P,
                                                        double2* __restrict__ A) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool active = j < n;
    const int64_t jj = active ? j : n - 1;
    const DerivUniform K = deriv_uniform<VAR>(P);
    const FarLane F = far_lane(panels[jj], K.s);
    const PanelBc bc = MODE == 1 ? bcs[jj] : rigid_bc();
    const int64_t i0 = (int64_t)blockIdx.y * rows_per_block;
    const int64_t i1 = min(n, i0 + rows_per_block);
    for (int64_t i = i0; i < i1; ++i) {
        double2 d_cb, d_hb = make_double2(0.0, 0.0), hb = make_double2(0.0, 0.0);
        far_sums_d<MODE, VAR>(F, sources[i], K, d_cb, d_hb, hb);
        const double2 out = deriv_from_blocks(d_cb, d_hb, hb, bc, P);
        if (active) A[i * lda + j] = out;
    }
}

// pairs_per_block near pairs per workgroup, lane per leaf as in near_kernel.
template <int MODE, int VAR>
__global__ __launch_bounds__(256) void near_deriv_kernel(const NearPair* __restrict__ pairs, int64_t npairs,
                                                         int pairs_per_block, const uint64_t* __restrict__ leaves,
                                                         const FarPanel* __restrict__ panels,
                                                         const Source* __restrict__ sources,
                                                         const PanelBc* __restrict__ bcs, int64_t lda,
                                                         DerivParams P, double2* __restrict__ A) {
    const int64_t p0 = (int64_t)blockIdx.x * pairs_per_block;
    const DerivUniform K = deriv_uniform<VAR>(P);
    near_pairs(
        pairs, p0, (int)min((int64_t)pairs_per_block, npairs - p0), leaves,
        [&](const NearPair& np, uint64_t code) {
            double2 d_cb, d_hb = make_double2(0.0, 0.0), hb = make_double2(0.0, 0.0);
            far_sums_d<MODE, VAR>(leaf_lane(panels[np.j], code, K.s), sources[np.i], K, d_cb, d_hb, hb);
            return deriv_from_blocks(d_cb, d_hb, hb, MODE == 1 ? bcs[np.j] : rigid_bc(), P);
        },
        [&](int, const NearPair& np, double2 v) { A[(int64_t)np.i * lda + np.j] = v; });
}

// One wave per panel: self-integral derivatives, free terms, BC free-term RHS.
__global__ __launch_bounds__(256) void self_deriv_kernel(const PanelGeom* __restrict__ geom,
                                                         const Source* __restrict__ sources,
                                                         const PanelBc* __restrict__ bcs, int general, int64_t n,
                                                         int64_t lda, DerivParams P, double2* __restrict__ A,
                                                         double2* __restrict__ rhs) {
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    const PanelBc bc = general ? bcs[i] : rigid_bc();
    const PanelGeom& G = geom[i];
    const Source S = sources[i];
    const double k2 = P.k * P.k;
    const SelfTier t = tier_for(P.k * G.size);
    const int ns = self_samples(t);
    Acc b = acc_zero(), d = acc_zero();
    for (int s = lane; s < ns; s += 64) self_sample_t<true>(G, t, s, S.c, S.n, P.wavruim, k2, P.k, P.hf, b, d);
    wave_sum_acc(b);
    wave_sum_acc(d);
    if (lane == 0) {
        double2 diag, local_rhs;
        deriv_free_terms(bc, P, &diag, &local_rhs);
        A[i * lda + i] = cadd(diag, deriv_coefficient(b, d, bc, P));
        rhs[i] = local_rhs;
    }
}

// Block per row: right-hand-side derivative over the nonzero-BC columns in a
// fixed order, as bc_rhs_kernel (4378 panels, 164 -> 81 us).
__global__ __launch_bounds__(256) void bc_rhs_deriv_kernel(const int32_t* __restrict__ cols, int64_t ncols,
                                                           const NearPair* __restrict__ pairs,
                                                           const int64_t* __restrict__ row_ptr,
                                                           const uint64_t* __restrict__ leaves,
                                                           const PanelGeom* __restrict__ geom,
                                                           const Source* __restrict__ sources,
                                                           const PanelBc* __restrict__ bcs, DerivParams P,
                                                           double2* __restrict__ rhs) {
    __shared__ double part[16][2];
    const int64_t i = blockIdx.x;
    const int group = threadIdx.x >> 4;
    const int lane = threadIdx.x & 15;
    const Source src = sources[i];
    const double k2 = P.k * P.k;
    double2 sum = make_double2(0.0, 0.0);
    const int64_t pb = row_ptr[i], pe = row_ptr[i + 1];
    for (int64_t c = group; c < ncols; c += 16) {
        const int32_t j = cols[c];
        const PanelGeom G = geom[j];
        Acc b = acc_zero(), d = acc_zero();
        if (j == i) {
            const SelfTier t = tier_for(P.k * G.size);
            const int ns = self_samples(t);
            for (int s = lane; s < ns; s += 16)
                self_sample_t<true>(G, t, s, src.c, src.n, P.wavruim, k2, P.k, P.hf, b, d);
        } else {
            int64_t lo = pb, hi = pe;
            while (lo < hi) {
                int64_t mid = (lo + hi) / 2;
                if (pairs[mid].j < j) lo = mid + 1; else hi = mid;
            }
            if (lo < pe && pairs[lo].j == j) {
                const NearPair np = pairs[lo];
                const int total = np.count * 13;
                for (int t = lane; t < total; t += 16) {
                    const int leaf = t / 13;
                    near_point_t<true>(G, leaves[np.begin + leaf], t - leaf * 13, src.c, src.n, P.wavruim, k2, P.k,
                                       P.hf, b, d);
                }
            } else if (lane < 13) {
                full_point_t<true>(G, lane, src.c, src.n, P.wavruim, k2, P.k, P.hf, b, d);
            }
        }
        row16_sum_acc(b);
        row16_sum_acc(d);
        sum = cadd(sum, deriv_bc_contribution(b, d, bcs[j], P));
    }
    if (lane == 0) {
        part[group][0] = sum.x;
        part[group][1] = sum.y;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double2 t = rhs[i];
        for (int w = 0; w < 16; ++w) t = cadd(t, make_double2(part[w][0], part[w][1]));
        rhs[i] = t;
    }
}

// Block per row: sum over nonzero-BC columns of tbem.rs:1419-1435, in a
// fixed order (sixteen lanes take columns g, g+16, ...; the groups summed in
// order).  FP64 issue bounds it: the rule's 13 points on 16 lanes leave 3 idle,
// on a wave 51 (4378 panels, 139 -> 82 us).
__global__ __launch_bounds__(256) void bc_rhs_kernel(const int32_t* __restrict__ cols, int64_t ncols,
                                                     const NearPair* __restrict__ pairs,
                                                     const int64_t* __restrict__ row_ptr,
                                                     const uint64_t* __restrict__ leaves,
                                                     const PanelGeom* __restrict__ geom,
                                                     const Source* __restrict__ sources,
                                                     const PanelBc* __restrict__ bcs, double k,
                                                     double wavruim, double tau_r, double2 beta,
                                                     double2 iwr, double2* __restrict__ rhs) {
    __shared__ double part[16][2];
    const int64_t i = blockIdx.x;
    const int group = threadIdx.x >> 4;
    const int lane = threadIdx.x & 15;
    const Source src = sources[i];
    const double k2 = k * k;
    const double2 gamma = make_double2(1.0, 0.0);
    const double2 tau = make_double2(tau_r, 0.0);
    double2 sum = make_double2(0.0, 0.0);
    const int64_t pb = row_ptr[i], pe = row_ptr[i + 1];
    for (int64_t c = group; c < ncols; c += 16) {
        const int32_t j = cols[c];
        const PanelGeom G = geom[j];
        Acc a = acc_zero();
        if (j == i) {
            const SelfTier t = tier_for(k * G.size);
            const int ns = self_samples(t);
            for (int s = lane; s < ns; s += 16) self_sample(G, t, s, src.c, src.n, wavruim, k2, a);
        } else {
            int64_t lo = pb, hi = pe;  // pairs of row i are sorted by column
            while (lo < hi) {
                int64_t mid = (lo + hi) / 2;
                if (pairs[mid].j < j) lo = mid + 1; else hi = mid;
            }
            if (lo < pe && pairs[lo].j == j) {
                const NearPair np = pairs[lo];
                const int total = np.count * 13;
                for (int t = lane; t < total; t += 16) {
                    int leaf = t / 13;
                    near_point(G, leaves[np.begin + leaf], t - leaf * 13, src.c, src.n, wavruim, k2, a);
                }
            } else if (lane < 13) {
                full_point(G, lane, src.c, src.n, wavruim, k2, a);
            }
        }
        row16_sum_acc(a);
        sum = cadd(sum, bc_contribution(a, bcs[j], gamma, tau, beta, iwr));
    }
    if (lane == 0) {
        part[group][0] = sum.x;
        part[group][1] = sum.y;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double2 t = rhs[i];
        for (int w = 0; w < 16; ++w) t = cadd(t, make_double2(part[w][0], part[w][1]));
        rhs[i] = t;
    }
}

// incident.rs:216-330, 807-834; bem_solver.rs:5005-5034 (reference order).
#pragma clang fp contract(off)
__device__ __forceinline__ double2 plane_wave_value(const Source& s, const double* d, double2 amp, double k,
                                                    double hf, double tau_r, double2 beta, double sign) {
    double kdotx = hf * k * (d[0] * s.c[0] + d[1] * s.c[1] + d[2] * s.c[2]);
    double kdotn = hf * k * (d[0] * s.n[0] + d[1] * s.n[1] + d[2] * s.n[2]);
    double sn, cs;
    sincos_red(kdotx, &sn, &cs);
    double2 p = cmul(amp, make_double2(cs, sn));
    double2 dpdn = cmul(make_double2(0.0, kdotn), p);
    double2 gp = cmul(make_double2(1.0, 0.0), p);
    double2 bt = cmul(beta, make_double2(tau_r, 0.0));
    double2 inc = cadd(gp, cmul(bt, dpdn));
    inc = make_double2(-inc.x, -inc.y);
    return cmul(inc, make_double2(sign, 0.0));
}

__global__ void plane_wave_kernel(const Source* __restrict__ sources, int64_t n,
                                  const double* __restrict__ dirs, const double2* __restrict__ amps,
                                  int64_t nrhs, double k, double hf, double tau_r, double2 beta,
                                  double sign, int accumulate, double2* __restrict__ rhs) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * nrhs) return;
    const int64_t i = t / nrhs;
    const int64_t c = t - i * nrhs;
    const double2 add = plane_wave_value(sources[i], dirs + 3 * c, amps[c], k, hf, tau_r, beta, sign);
    rhs[t] = accumulate ? cadd(rhs[t], add) : add;
}

#pragma clang fp contract(on)

// Far entries of a frequency family (instances on one mesh with wavenumbers
// k_f = k0 + f dk): one lane per column, FAMILY_ROWS rows per workgroup,
// blockIdx.z the family.  Per TR13 point the k-independent geometry
// (distance, 1/r, normal projections, weight) is formed once, the phase
// exp(i k0 r) and the step exp(i dk r) come from two sincos evaluations, and
// each member then needs only the phase advance (one complex product) and
// its channel sums.  The members' own k_f enter the channel formulas; the
// phase recurrence differs from a direct sincos(k_f r) by at most about
// F ulp of the phase (F <= 16).  Velocity panels without admittance:
// A_ij = H tau + E beta (velocity_coefficient) from separate sums of the H and E
// channels per member, 15 FP64 instructions a member and evaluation, over the
// distances of family_points; far_sums folds tau and beta into one weight and
// takes its geometry and phases from the panel centre.
constexpr int FAMILY_ROWS = 16;

template <int F>
__global__ __launch_bounds__(256) void batch_far_family_kernel(const FreqFamily* __restrict__ families,
                                                               const BatchInstance* __restrict__ inst,
                                                               const FarPanel* __restrict__ far,
                                                               const Source* __restrict__ sources,
                                                               double2* __restrict__ A) {
    const FreqFamily& fam = families[blockIdx.z];
    const int64_t n = fam.n;
    const int64_t i0 = (int64_t)blockIdx.y * FAMILY_ROWS;
    if ((int64_t)blockIdx.x * 256 >= n || i0 >= n) return;
    const int count = fam.count;
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool active = j < n;
    const FarPanel P = far[fam.panel_off + (active ? j : n - 1)];
    const FamilyPoints FP = family_points(P);
    const Source* src = sources + fam.panel_off;
    const double k0 = fam.k0, dk = fam.dk;
    const int64_t i1 = min(n, i0 + (int64_t)FAMILY_ROWS);
    for (int64_t i = i0; i < i1; ++i) {
        const Source S = src[i];
        const double rel0 = P.v0[0] - S.c[0];
        const double rel1 = P.v0[1] - S.c[1];
        const double rel2 = P.v0[2] - S.c[2];
        const double nxny = S.n[0] * P.nf[0] + S.n[1] * P.nf[1] + S.n[2] * P.nf[2];
        const double a = rel0 * rel0 + rel1 * rel1 + rel2 * rel2;
        const double b1 = 2.0 * (rel0 * P.e1[0] + rel1 * P.e1[1] + rel2 * P.e1[2]);
        const double b2 = 2.0 * (rel0 * P.e2[0] + rel1 * P.e2[1] + rel2 * P.e2[2]);
        const double pr = rel0 * P.nf[0] + rel1 * P.nf[1] + rel2 * P.nf[2];
        const double g0 = -(rel0 * S.n[0] + rel1 * S.n[1] + rel2 * S.n[2]);
        const double g1 = -(P.e1[0] * S.n[0] + P.e1[1] * S.n[1] + P.e1[2] * S.n[2]);
        const double g2 = -(P.e2[0] * S.n[0] + P.e2[1] * S.n[1] + P.e2[2] * S.n[2]);
        double hr[F], hi[F], er[F], ei[F];
#pragma unroll
        for (int f = 0; f < F; ++f) hr[f] = hi[f] = er[f] = ei[f] = 0.0;
#pragma clang loop unroll(disable)
        for (int q = 0; q < 13; ++q) {
            const double sq = kTrS[q], tq = kTrT[q];
            const double u1 = __builtin_fma(tq, FP.e12x2, __builtin_fma(sq, FP.e11, b1));
            const double u2 = __builtin_fma(tq, FP.e22, b2);
            const double d2 = fmax(__builtin_fma(sq, u1, __builtin_fma(tq, u2, a)), 1e-300);
            const double inv = rsqrt_nr(d2);
            const double dis = d2 * inv;
            const double pn = pr * inv;                                                // r^.n_y
            const double qn = __builtin_fma(sq, g1, __builtin_fma(tq, g2, g0)) * inv;  // -r^.n_x
            const double re2 = (kTrW[q] * P.wj) * inv;
            const double inv2 = inv * inv;
            const double rq = pn * qn;
            // ef = (3/r^2 - k^2) rq + n.n/r^2  -  i k (3 rq + n.n)/r
            const double ef0 = (3.0 * inv2) * rq + nxny * inv2;
            const double ef1 = -inv * (3.0 * rq + nxny);
            // member f, phase p = exp(i k_f r): H += p re2 pn (-1/r + i k_f),
            // E += p re2 (ef0 - k_f^2 rq + i k_f ef1); the k_f-free factors once here
            const double wb = re2 * pn, wa = -wb * inv;
            const double E0 = re2 * ef0, R = re2 * rq, E1 = re2 * ef1;
            double phr, phi, str, sti;
            sincos_red(k0 * dis, &phi, &phr);
            sincos_red(dk * dis, &sti, &str);
            // all F members, also past count (kf = 0 there; those sums are dropped)
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const double kf = fam.kf[f];
                const double u = __builtin_fma(-kf * kf, R, E0);
                const double v = kf * E1;
                const double t = kf * wb;
                hr[f] = __builtin_fma(-phi, t, __builtin_fma(phr, wa, hr[f]));
                hi[f] = __builtin_fma(phr, t, __builtin_fma(phi, wa, hi[f]));
                er[f] = __builtin_fma(-phi, v, __builtin_fma(phr, u, er[f]));
                ei[f] = __builtin_fma(phi, u, __builtin_fma(phr, v, ei[f]));
                const double nr = __builtin_fma(phr, str, -phi * sti);
                phi = __builtin_fma(phr, sti, phi * str);
                phr = nr;
            }
        }
        if (active) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                if (f < count) {
                    const BatchInstance& I = inst[fam.member[f]];
                    A[I.a_off + i * n + j] =
                        velocity_coefficient(hr[f], hi[f], er[f], ei[f], I.tau, make_double2(I.beta[0], I.beta[1]));
                }
            }
        }
    }
}

// Near pairs of a frequency family: the subdivided-leaf quadrature of each
// pair (regular.rs:164-281, the points of near_point) with the point geometry
// formed once for all members.  Sixteen lanes take one pair (a wave four),
// lanes over (leaf, point); per point the phase exp(i k0 r) and the step
// exp(i dk r) come from two sincos evaluations and each member advances the
// phase by one complex product.  Rigid panels need the H and E channels
// only; the 16-lane sums use row DPP, and lane f writes member f's entry.
constexpr int NEAR_FAMILY_LANES = 16;

template <int F>
__global__ __launch_bounds__(256) void batch_near_family_kernel(const FreqFamily* __restrict__ families,
                                                                const BatchInstance* __restrict__ inst,
                                                                const NearPair* __restrict__ pairs,
                                                                const uint64_t* __restrict__ leaves,
                                                                const PanelGeom* __restrict__ geom,
                                                                const Source* __restrict__ sources,
                                                                double2* __restrict__ A) {
#pragma clang fp contract(on)
    const FreqFamily& fam = families[blockIdx.y];
    const int sub = threadIdx.x & (NEAR_FAMILY_LANES - 1);
    const int count = fam.count;
    const double k0 = fam.k0, dk = fam.dk;
    const int64_t n = fam.n;
    const int64_t step = (int64_t)gridDim.x * (256 / NEAR_FAMILY_LANES);
    for (int64_t p = (int64_t)blockIdx.x * (256 / NEAR_FAMILY_LANES) + (threadIdx.x / NEAR_FAMILY_LANES);
         p < fam.npairs; p += step) {
        const NearPair np = pairs[fam.pair_begin + p];
        const PanelGeom G = geom[fam.panel_off + np.j];
        const Source S = sources[fam.panel_off + np.i];
        const double nxny = S.n[0] * G.nf[0] + S.n[1] * G.nf[1] + S.n[2] * G.nf[2];
        double hr[F], hi[F], er[F], ei[F];
#pragma unroll
        for (int f = 0; f < F; ++f) hr[f] = hi[f] = er[f] = ei[f] = 0.0;
        const int total = np.count * 13;
        for (int t = sub; t < total; t += NEAR_FAMILY_LANES) {
            const int leaf = t / 13;
            const int q = t - leaf * 13;
            double xi[3], et[3];
            decode_leaf(leaves[np.begin + leaf], xi, et);
            const double cs = kTrS[q], ec = kTrT[q];
            const double l0 = 1.0 - cs - ec;
            const double xio = xi[0] * l0 + xi[1] * cs + xi[2] * ec;
            const double eto = et[0] * l0 + et[1] * cs + et[2] * ec;
            const double det = fabs((xi[1] - xi[0]) * (et[2] - et[0]) - (xi[2] - xi[0]) * (et[1] - et[0]));
            const double wga = ((kTrW[q] * 0.5) * det) * G.jac;
            double pos[3];
            shape_pos(G.c, xio, eto, pos);
            const double d0 = pos[0] - S.c[0], d1 = pos[1] - S.c[1], d2 = pos[2] - S.c[2];
            const double dsq = d0 * d0 + d1 * d1 + d2 * d2;
            if (!(dsq > 1e-30)) continue;  // the point evaluation skips |d| <= 1e-15
            const double inv = rsqrt_nr(dsq);
            const double dis = dsq * inv;
            const double u0 = d0 * inv, u1 = d1 * inv, u2 = d2 * inv;
            const double re2 = (wga * (1.0 / FOUR_PI)) * inv;
            const double pn = u0 * G.nf[0] + u1 * G.nf[1] + u2 * G.nf[2];   // r^.n_y
            const double qn = -(u0 * S.n[0] + u1 * S.n[1] + u2 * S.n[2]);  // -r^.n_x
            const double rq = pn * qn;
            const double inv2 = inv * inv;
            const double ef0 = (3.0 * inv2) * rq + nxny * inv2;
            const double ef1 = -inv * (3.0 * rq + nxny);
            // the channel factors of batch_far_family_kernel
            const double wb = re2 * pn, wa = -wb * inv;
            const double E0 = re2 * ef0, R = re2 * rq, E1 = re2 * ef1;
            double phr, phi, str, sti;
            sincos_red(k0 * dis, &phi, &phr);
            sincos_red(dk * dis, &sti, &str);
            // all F members, also past count (kf = 0 there; those sums are dropped)
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const double kf = fam.kf[f];
                const double u = E0 - (kf * kf) * R;
                const double v = kf * E1;
                const double t = kf * wb;
                hr[f] += phr * wa - phi * t;
                hi[f] += phi * wa + phr * t;
                er[f] += phr * u - phi * v;
                ei[f] += phr * v + phi * u;
                const double nr = phr * str - phi * sti;
                phi = phr * sti + phi * str;
                phr = nr;
            }
        }
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if (f < count) {
                const double h_r = row16_sum(hr[f]), h_i = row16_sum(hi[f]);
                const double e_r = row16_sum(er[f]), e_i = row16_sum(ei[f]);
                if (sub == f) {
                    const BatchInstance& I = inst[fam.member[f]];
                    const double tau = I.tau;
                    A[I.a_off + (int64_t)np.i * n + np.j] =
                        make_double2(h_r * tau + (e_r * I.beta[0] - e_i * I.beta[1]),
                                     h_i * tau + (e_r * I.beta[1] + e_i * I.beta[0]));
                }
            }
        }
    }
}

// Batch of rigid instances, two persistent launches over the same items
// (instance, first row); the host orders items by decreasing instance size
// and each workgroup takes items from a counter until none are left.
// PHASE 0 writes the far entries of the item's rows (lane per column) and
// their plane-wave right-hand sides; PHASE 1, launched after it, overwrites
// the near pairs and the diagonal of those rows, which is the overwrite order
// of the single-system launch.  The phases are separate kernels because the
// near/self code needs 201 registers, two waves to a SIMD, and the far loop 147,
// three.
template <int PHASE>
__global__ __launch_bounds__(256) void batch_assemble_kernel(BatchAssemblyArgs args) {
    __shared__ int s_item;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    for (;;) {
        if (threadIdx.x == 0) s_item = (int)atomicAdd(args.counter + PHASE, 1u);
        __syncthreads();
        const int it = s_item;
        __syncthreads();
        if (it >= args.nitems) break;
        const int2 item = args.items[it];
        const BatchInstance& I = args.inst[item.x];
        const int64_t n = I.n;
        const int64_t r0 = item.y;
        const int64_t r1 = min(n, r0 + (int64_t)args.rows_per_item);
        const Source* src = args.src + I.panel_off;
        double2* A = args.A + I.a_off;
        const double k = I.k;
        const double2 beta = make_double2(I.beta[0], I.beta[1]);
        if (PHASE == 0) {
            const FarPanel* far = args.far + I.panel_off;
            auto fill = [&](auto variant) {
                constexpr int VAR = decltype(variant)::value;
                const FarUniform K = far_uniform<VAR>(k, I.tau, beta);
                for (int64_t jc = 0; jc < n; jc += 256) {
                    const int64_t j = jc + threadIdx.x;
                    const bool active = j < n;
                    const FarLane P = far_lane(far[active ? j : n - 1], K.s);
                    for (int64_t i = r0; i < r1; ++i) {
                        const double2 v = far_entry<0, VAR>(P, src[i], PanelBc(), K, make_double2(0.0, 0.0));
                        if (active) A[i * n + j] = v;
                    }
                }
            };
            // members of a frequency family got their far entries from batch_far_family_kernel
            if (!I.in_family) {
                if (I.far_variant == FAR_SHORT)
                    fill(std::integral_constant<int, FAR_SHORT>());
                else if (I.far_variant == FAR_LONG)
                    fill(std::integral_constant<int, FAR_LONG>());
                else
                    fill(std::integral_constant<int, FAR_GENERAL>());
            }
            const int64_t nr = (r1 - r0) * I.ncol;
            for (int64_t t = threadIdx.x; t < nr; t += 256) {
                const int64_t i = r0 + t / I.ncol;
                const int c = (int)(t % I.ncol);
                args.rhs[I.vec_off + i * I.ncol + c] = plane_wave_value(
                    src[i], args.dirs + 3 * (I.dir_off + c), make_double2(1.0, 0.0), k, 1.0, I.tau, beta, I.sign);
            }
        } else {
            const PanelGeom* geom = args.geom + I.panel_off;
            const FarPanel* far = args.far + I.panel_off;
            const PanelBc bc = rigid_bc();
            const double2 iwr = make_double2(0.0, 0.0);  // no admittance on rigid panels
            // members of a frequency family got their near pairs from batch_near_family_kernel
            const int64_t pb = args.row_ptr[I.panel_off + r0];
            const int64_t pe = I.in_family ? pb : args.row_ptr[I.panel_off + r1];
            auto fill = [&](auto variant) {
                constexpr int VAR = decltype(variant)::value;
                const FarUniform K = far_uniform<VAR>(k, I.tau, beta);
                for (int64_t p = pb; p < pe; p += 256)
                    near_pairs(
                        args.pairs, p, (int)min((int64_t)256, pe - p), args.leaves,
                        [&](const NearPair& np, uint64_t code) {
                            return far_entry<0, VAR>(leaf_lane(far[np.j], code, K.s), src[np.i], bc, K, iwr);
                        },
                        [&](int, const NearPair& np, double2 v) { A[(int64_t)np.i * n + np.j] = v; });
            };
            if (I.far_variant == FAR_SHORT)
                fill(std::integral_constant<int, FAR_SHORT>());
            else if (I.far_variant == FAR_LONG)
                fill(std::integral_constant<int, FAR_LONG>());
            else
                fill(std::integral_constant<int, FAR_GENERAL>());
            for (int64_t i = r0 + wave; i < r1; i += 4) {
                double2 diag, unused;
                self_entry(geom[i], src[i], bc, k, k, I.tau, beta, iwr, lane, &diag, &unused);
                if (lane == 0) A[i * n + i] = diag;
            }
        }
    }
}

__global__ void reset_counters_kernel(unsigned* counter) { counter[threadIdx.x] = 0u; }

// ---------------------------------------------------------------------------
// Matrix-free exact product y = sign * A x (apply_tbem_stabilized_exact,
// crates/sonium-bem/src/core/assembly/hmatrix.rs:2363-2425) with the entries of
// the assembly kernels, evaluated on the fly in O(N) memory:
//   exact_far_kernel   far[i] = sum over j != i of the 13-point entry times x_j
//                      (lane per column, EXACT_ROWS rows per workgroup, row sums
//                      reduced across the workgroup in a fixed order);
//   exact_near_kernel  per near pair: (subdivided entry - 13-point entry) x_j;
//   exact_self_kernel  per panel: diagonal entry times x_i;
//   exact_combine_kernel  y_i = sign (far_i + near pairs of row i in CSR
//                      order + self_i).
constexpr int EXACT_ROWS = 4;

template <int MODE, int VAR>
__global__ __launch_bounds__(256) void exact_far_kernel(const FarPanel* __restrict__ panels,
                                                        const Source* __restrict__ sources,
                                                        const PanelBc* __restrict__ bcs, int64_t n, double k,
                                                        double tau_r, double2 beta, double2 iwr,
                                                        const double2* __restrict__ x, double2* __restrict__ out) {
    __shared__ double2 sums[EXACT_ROWS][256];  // each lane's row sums
    __shared__ double2 red[4][EXACT_ROWS];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * EXACT_ROWS;
    const FarUniform K = far_uniform<VAR>(k, tau_r, beta);
    for (int r = 0; r < EXACT_ROWS; ++r) sums[r][threadIdx.x] = make_double2(0.0, 0.0);
    // a column chunk's panel constants serve all rows; the rows run one after
    // another, so one row's points are live at a time
    for (int64_t jc = 0; jc < n; jc += 256) {
        const int64_t j = jc + threadIdx.x;
        const bool active = j < n;
        const int64_t jj = active ? j : n - 1;
        const FarLane P = far_lane(panels[jj], K.s);
        PanelBc bc;
        if (MODE == 1) bc = bcs[jj];
        const double2 xj = x[jj];
#pragma clang loop unroll(disable)
        for (int r = 0; r < EXACT_ROWS; ++r) {
            const int64_t i = min(i0 + r, n - 1);  // rows past n are computed and dropped
            const double2 v = far_entry<MODE, VAR>(P, sources[i], bc, K, iwr);
            if (active && j != i) {
                double2 acc = sums[r][threadIdx.x];
                acc.x += v.x * xj.x - v.y * xj.y;
                acc.y += v.x * xj.y + v.y * xj.x;
                sums[r][threadIdx.x] = acc;
            }
        }
    }
    for (int r = 0; r < EXACT_ROWS; ++r) {
        double2 acc = sums[r][threadIdx.x];
        acc.x = wave_sum(acc.x);
        acc.y = wave_sum(acc.y);
        if (lane == 0) red[wave][r] = acc;
    }
    __syncthreads();
    if (threadIdx.x < EXACT_ROWS && i0 + threadIdx.x < n) {
        double2 t = red[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) t = cadd(t, red[w][threadIdx.x]);
        out[i0 + threadIdx.x] = t;
    }
}

template <int MODE, int VAR>
__global__ __launch_bounds__(256) void exact_near_kernel(const NearPair* __restrict__ pairs, int64_t npairs,
                                                         int pairs_per_block, const uint64_t* __restrict__ leaves,
                                                         const FarPanel* __restrict__ panels,
                                                         const Source* __restrict__ sources,
                                                         const PanelBc* __restrict__ bcs, double k, double tau_r,
                                                         double2 beta, double2 iwr, const double2* __restrict__ x,
                                                         double2* __restrict__ out) {
    const int64_t p0 = (int64_t)blockIdx.x * pairs_per_block;
    const FarUniform K = far_uniform<VAR>(k, tau_r, beta);
    near_pairs(
        pairs, p0, (int)min((int64_t)pairs_per_block, npairs - p0), leaves,
        [&](const NearPair& np, uint64_t code) {
            PanelBc bc;
            if (MODE == 1) bc = bcs[np.j];
            return far_entry<MODE, VAR>(leaf_lane(panels[np.j], code, K.s), sources[np.i], bc, K, iwr);
        },
        [&](int t, const NearPair& np, double2 v) {
            PanelBc bc;
            if (MODE == 1) bc = bcs[np.j];
            const double2 f = far_entry<MODE, VAR>(far_lane(panels[np.j], K.s), sources[np.i], bc, K, iwr);
            out[p0 + t] = cmul(csub(v, f), x[np.j]);
        });
}

__global__ __launch_bounds__(256) void exact_self_kernel(const PanelGeom* __restrict__ geom,
                                                         const Source* __restrict__ sources,
                                                         const PanelBc* __restrict__ bcs, int general, int64_t n,
                                                         double k, double wavruim, double tau_r, double2 beta,
                                                         double2 iwr, const double2* __restrict__ x,
                                                         double2* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    const PanelBc bc = general ? bcs[i] : rigid_bc();
    double2 diag, unused;
    self_entry(geom[i], sources[i], bc, k, wavruim, tau_r, beta, iwr, lane, &diag, &unused);
    if (lane == 0) out[i] = cmul(diag, x[i]);
}

__global__ void exact_combine_kernel(const double2* __restrict__ far, const double2* __restrict__ near,
                                     const int64_t* __restrict__ row_ptr, const double2* __restrict__ self,
                                     int64_t n, double sign, double2* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double2 s = far[i];
    for (int64_t p = row_ptr[i]; p < row_ptr[i + 1]; ++p) s = cadd(s, near[p]);
    s = cadd(s, self[i]);
    y[i] = make_double2(sign * s.x, sign * s.y);
}

// ---------------------------------------------------------------------------
// Pressure at evaluation points (compute_scattered_field / compute_total_field,
// crates/sonium-bem/src/core/postprocess/pressure.rs:1388-1480, 1566-1620,
// 1987-2044), constant basis on Tri3 panels:
//   p(x) = sum_j sum_q [p_j G (-1/r + ik) (r.n_j)/r - v_j i rho omega G] J_j w_q
// with r = y_q - x, G = e^{ikr}/(4 pi r) and the 7-point rule.  A workgroup
// takes FIELD_ROWS points and one slice of the panels (lane per panel); the
// points' coordinates are wave-uniform.  The slices' partial sums are added per
// point in slice order.
//
// FP64 VALU issue bounds it.  Distances come from the panel's corner offsets
// and phases from its centre (far_sums): the rule's points are c, c + kappa V_i
// and c + kappa' V_i, so an evaluation takes 29 FP64 instructions (42 with the
// pair's share) where a difference per point and a reduced sine took 65, and
// 5000 points x 10240 panels take 640 us instead of 904.  Within two panel
// radii of a panel the expansion of the distance would lose digits, so there
// the lanes take the differences directly (field_near), which also leaves out
// a quadrature point that the evaluation point sits on.
constexpr int FIELD_ROWS = 8;
// TR7 (gauss.rs:516-524); weights are used times 0.5
constexpr double TR7_K1 = 0.797426985353087 - 0.101286507323456;
constexpr double TR7_K2 = 0.059715871789770 - 0.470142064105115;
constexpr double TR7_W0 = 0.225, TR7_W1 = 0.125939180544827, TR7_W2 = 0.132394152788506;

// sum w z (-1/r + ik) dr/dn and sum w z of one pair without the panel factor.
// A wave with a close panel waits for the whole chain, so the points are unrolled, with their constants as literals
// and one load of the panel, and each lane takes its own close rows: 50 points off 320 panels 65 us where a loop
// over tables and all rows took 77 (57 away from the panels).
__device__ __forceinline__ void field_near(const FarPanel& P, const double* x, double k, double2* h, double2* g) {
    constexpr double S[7] = {0.333333333333333, 0.797426985353087, 0.101286507323456, 0.101286507323456,
                             0.470142064105115, 0.059715871789770, 0.470142064105115};
    constexpr double T[7] = {0.333333333333333, 0.101286507323456, 0.797426985353087, 0.101286507323456,
                             0.059715871789770, 0.470142064105115, 0.470142064105115};
    double v0[3], e1[3], e2[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v0[c] = P.v0[c];
        e1[c] = P.e1[c];
        e2[c] = P.e2[c];
    }
    const double xr[3] = {x[0], x[1], x[2]};
    const double pr = (v0[0] - xr[0]) * P.nf[0] + (v0[1] - xr[1]) * P.nf[1] + (v0[2] - xr[2]) * P.nf[2];
    double hx = 0.0, hy = 0.0, gx = 0.0, gy = 0.0;
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        const double wq = q == 0 ? TR7_W0 : q < 4 ? TR7_W1 : TR7_W2;
        double d[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) d[c] = __builtin_fma(S[q], e1[c], __builtin_fma(T[q], e2[c], v0[c])) - xr[c];
        const double d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        const bool off = d2 > 1e-30;  // a point within 1e-15 of the quadrature point contributes nothing
        const double inv = rsqrt_nr(off ? d2 : 1.0);
        double sn, cs;
        sincos_red(k * (d2 * inv), &sn, &cs);
        const double w = off ? wq * inv : 0.0;
        const double zr = cs * w, zi = sn * w;
        const double drdn = pr * inv;
        hx += (-zr * inv - zi * k) * drdn;
        hy += (zr * k - zi * inv) * drdn;
        gx += zr;
        gy += zi;
        asm volatile("" : "+v"(v0[0]), "+v"(hx), "+v"(hy), "+v"(gx), "+v"(gy));  // one point at a time
    }
    *h = make_double2(hx, hy);
    *g = make_double2(gx, gy);
}

template <int HAS_V, int VAR>
__global__ __launch_bounds__(256) void field_kernel(const FarPanel* __restrict__ panels, int64_t n,
                                                    const double* __restrict__ points, int64_t m,
                                                    const double2* __restrict__ p, const double2* __restrict__ v,
                                                    double k, double pf, int64_t panels_per_slice,
                                                    double2* __restrict__ part) {
    __shared__ double2 red[4][FIELD_ROWS];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * FIELD_ROWS;
    const int64_t jbeg = (int64_t)blockIdx.y * panels_per_slice;
    const int64_t jend = min(n, jbeg + panels_per_slice);
    const double s = VAR == FAR_GENERAL ? 1.0 : k, kap = VAR == FAR_GENERAL ? k : 1.0;
    double2 acc[FIELD_ROWS];
#pragma unroll
    for (int r = 0; r < FIELD_ROWS; ++r) acc[r] = make_double2(0.0, 0.0);
    for (int64_t jc = jbeg; jc < jend; jc += 256) {
        const int64_t j = jc + threadIdx.x;
        const bool active = j < jend;
        const FarPanel& P = panels[active ? j : n - 1];
        const double2 pj = p[active ? j : n - 1];
        const double2 vj = HAS_V ? v[active ? j : n - 1] : make_double2(0.0, 0.0);
        const FarLane F = far_lane(P, s);
        const double scale = (active && F.wj > 0.0) ? F.wj : 0.0;  // w J / (4 pi), times 0.5 for the rule
        const double reach = 4.0 * fmax(F.L[0], fmax(F.L[1], F.L[2]));
        unsigned close = 0;  // rows within reach of this lane's panel
        // p_j h - i pf v_j g
        auto term = [&](double2 h, double2 g) {
            double2 t = make_double2(scale * __builtin_fma(pj.x, h.x, -pj.y * h.y),
                                     scale * __builtin_fma(pj.x, h.y, pj.y * h.x));
            if (HAS_V) {
                const double sp = scale * pf;
                t.x = __builtin_fma(sp, __builtin_fma(vj.x, g.y, vj.y * g.x), t.x);
                t.y = __builtin_fma(sp, __builtin_fma(vj.y, g.y, -vj.x * g.x), t.y);
            }
            return t;
        };
#pragma unroll
        for (int r = 0; r < FIELD_ROWS; ++r) {
            const double* xr = points + 3 * min(i0 + r, m - 1);  // rows past m are computed and dropped
            double x[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                x[d] = (F.v0[d] - xr[d]) + F.cv[d];
                if (VAR != FAR_GENERAL) x[d] *= s;
            }
            const double A = dot3(x, x);
            const double D1 = dot3(x, F.V1), D2 = dot3(x, F.V2);
            const double D[3] = {-(D1 + D2), D1, D2};
            const double pr = dot3(x, F.nf);
            const double yc = rsqrt_nr(A);
            const double rc = A * yc;
            struct Part {
                double hr, hi, gr, gi;
            };
            double Ap = A;
            auto point = [&](double d2, bool centre, Part& a) {
                const double y = rsqrt_nr(d2);
                const double u = y * y;
                const double uy = u * y;
                double sn = 0.0, cs = 1.0;
                if (!centre)
                    sincos_difference<VAR>(VAR == FAR_GENERAL ? kap * __builtin_fma(d2, y, -rc)
                                                              : __builtin_fma(d2, y, -rc), &sn, &cs);
                const double ku = VAR == FAR_GENERAL ? kap * u : u;
                a.hr = __builtin_fma(-cs, uy, a.hr);
                a.hi = __builtin_fma(cs, ku, a.hi);
                if (!centre) {
                    a.hr = __builtin_fma(-sn, ku, a.hr);
                    a.hi = __builtin_fma(-sn, uy, a.hi);
                }
                if (HAS_V) {
                    a.gr = __builtin_fma(cs, y, a.gr);
                    if (!centre) a.gi = __builtin_fma(sn, y, a.gi);
                    asm volatile("" : "+v"(Ap), "+v"(a.hr), "+v"(a.hi), "+v"(a.gr), "+v"(a.gi));
                } else {
                    asm volatile("" : "+v"(Ap), "+v"(a.hr), "+v"(a.hi));  // one point at a time, as in far_sums
                }
            };
            Part tot = {0.0, 0.0, 0.0, 0.0};
            auto add = [&](double w, const Part& a) {
                tot.hr = __builtin_fma(w, a.hr, tot.hr);
                tot.hi = __builtin_fma(w, a.hi, tot.hi);
                if (HAS_V) {
                    tot.gr = __builtin_fma(w, a.gr, tot.gr);
                    tot.gi = __builtin_fma(w, a.gi, tot.gi);
                }
            };
            Part a0 = {0.0, 0.0, 0.0, 0.0}, a1 = a0, a2 = a0;
            point(A, true, a0);
            add(TR7_W0, a0);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                point(__builtin_fma(TR7_K1 * TR7_K1, F.L[i], __builtin_fma(2.0 * TR7_K1, D[i], Ap)), false, a1);
            add(TR7_W1, a1);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                point(__builtin_fma(TR7_K2 * TR7_K2, F.L[i], __builtin_fma(2.0 * TR7_K2, D[i], Ap)), false, a2);
            add(TR7_W2, a2);
            double sn, cs;
            sincos_red(VAR == FAR_GENERAL ? kap * rc : rc, &sn, &cs);
            const double fh = (s * s) * pr;
            double2 h = make_double2(fh * __builtin_fma(cs, tot.hr, -sn * tot.hi),
                                     fh * __builtin_fma(cs, tot.hi, sn * tot.hr));
            double2 g = make_double2(0.0, 0.0);
            if (HAS_V)
                g = make_double2(s * __builtin_fma(cs, tot.gr, -sn * tot.gi),
                                 s * __builtin_fma(cs, tot.gi, sn * tot.gr));
            const double2 t = term(h, g);
            const bool far = A > reach;
            if (!far) close |= 1u << r;
            acc[r].x += far ? t.x : 0.0;
            acc[r].y += far ? t.y : 0.0;
        }
        // each lane its own close rows: few, and rarely the same as its neighbours'
#pragma clang loop unroll(disable)
        for (unsigned left = close; left; left &= left - 1) {
            const int r = __builtin_ctz(left);
            double2 h, g;
            field_near(P, points + 3 * min(i0 + r, m - 1), k, &h, &g);
            const double2 t = term(h, g);
#pragma unroll
            for (int q = 0; q < FIELD_ROWS; ++q) {
                acc[q].x += q == r ? t.x : 0.0;
                acc[q].y += q == r ? t.y : 0.0;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < FIELD_ROWS; ++r) {
        acc[r].x = wave_sum(acc[r].x);
        acc[r].y = wave_sum(acc[r].y);
        if (lane == 0) red[wave][r] = acc[r];
    }
    __syncthreads();
    if (threadIdx.x < FIELD_ROWS && i0 + threadIdx.x < m) {
        double2 t = red[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) t = cadd(t, red[w][threadIdx.x]);
        part[(int64_t)blockIdx.y * m + i0 + threadIdx.x] = t;
    }
}

// Incident pressure and normal derivative of one source at x with normal nx
// (incident.rs:216-420); n == nullptr skips the derivative.  Reference
// operation order, as plane_wave_value.
#pragma clang fp contract(off)
__device__ inline void incident_value(const IncidentSource& s, const double* x, const double* nx, double k, double hf,
                                      double2* p, double2* dpdn) {
    const double2 amp = make_double2(s.amp[0], s.amp[1]);
    if (s.kind == 0) {
        double sn, cs;
        sincos_red(hf * k * (s.v[0] * x[0] + s.v[1] * x[1] + s.v[2] * x[2]), &sn, &cs);
        *p = cmul(amp, make_double2(cs, sn));
        if (nx) *dpdn = cmul(make_double2(0.0, hf * k * (s.v[0] * nx[0] + s.v[1] * nx[1] + s.v[2] * nx[2])), *p);
        return;
    }
    const double dx = x[0] - s.v[0], dy = x[1] - s.v[1], dz = x[2] - s.v[2];
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    *p = make_double2(0.0, 0.0);
    if (nx) *dpdn = make_double2(0.0, 0.0);
    if (!(r > 1e-10)) return;
    double sn, cs;
    sincos_red(hf * k * r, &sn, &cs);
    const double w = 1.0 / (12.566370614359172 * r);
    const double2 g = make_double2(cs * w, sn * w);
    *p = cmul(amp, g);
    if (nx) {
        const double2 dgdr = cmul(make_double2(-1.0 / r, hf * k), g);
        const double drdn = (dx * nx[0] + dy * nx[1] + dz * nx[2]) / r;
        *dpdn = cmul(amp, cscale(dgdr, drdn));
    }
}

// rhs_i (+)= sign * -(gamma p_inc + beta tau dp_inc/dn) over the sources in order.
__global__ void source_rhs_kernel(const Source* __restrict__ centers, int64_t n, const IncidentSource* __restrict__ srcs,
                                  int64_t nsrc, double k, double hf, double tau_r, double2 beta, double sign,
                                  int accumulate, double2* __restrict__ rhs) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Source c = centers[i];
    double2 p = make_double2(0.0, 0.0), q = make_double2(0.0, 0.0);
    for (int64_t w = 0; w < nsrc; ++w) {
        double2 pw, qw;
        incident_value(srcs[w], c.c, c.n, k, hf, &pw, &qw);
        p = cadd(p, pw);
        q = cadd(q, qw);
    }
    // incident.rs:825-831 and bem_solver.rs:5005-5034, as plane_wave_value
    double2 inc = cadd(cmul(make_double2(1.0, 0.0), p), cmul(cmul(beta, make_double2(tau_r, 0.0)), q));
    inc = make_double2(-inc.x, -inc.y);
    inc = cmul(inc, make_double2(sign, 0.0));
    rhs[i] = accumulate ? cadd(rhs[i], inc) : inc;
}
#pragma clang fp contract(on)

// scattered[i] = sum over slices of the partials; incident[i] = plane waves at
// x_i (incident.rs:216-260); total[i] = incident + scattered (FieldPoint::new,
// pressure.rs:32-41).  incident and total may be null.
__global__ void field_finish_kernel(const double2* __restrict__ part, int slices, const double* __restrict__ points,
                                    int64_t m, const IncidentSource* __restrict__ srcs, int64_t nsrc, double k,
                                    double hf, double2* __restrict__ scattered, double2* __restrict__ incident,
                                    double2* __restrict__ total) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    double2 s = make_double2(0.0, 0.0);
    for (int z = 0; z < slices; ++z) s = cadd(s, part[(int64_t)z * m + i]);
    scattered[i] = s;
    if (!incident && !total) return;
    double2 inc = make_double2(0.0, 0.0);
    for (int64_t w = 0; w < nsrc; ++w) {
        double2 p, unused;
        incident_value(srcs[w], points + 3 * i, nullptr, k, hf, &p, &unused);
        inc = cadd(inc, p);
    }
    if (incident) incident[i] = inc;
    if (total) total[i] = cadd(inc, s);
}

// Surface Cauchy data of each panel from its BC when no velocity is given
// (constant_cauchy_data, pressure.rs:1481-1520): velocity panels (sol, value),
// admittance panels (sol, value + adm sol), pressure panels
// (value - p_inc(c), (sol - dp_inc/dn(c)) / (i pf)) with the plane waves at the
// collocation point.
__global__ void field_cauchy_kernel(const PanelBc* __restrict__ bcs, const Source* __restrict__ src,
                                    const double2* __restrict__ sol, int64_t n, const IncidentSource* __restrict__ srcs,
                                    int64_t nsrc, double k, double hf, double pf, double2* __restrict__ pe,
                                    double2* __restrict__ ve) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const PanelBc bc = bcs[j];
    const double2 s = sol[j];
    const double2 val = make_double2(bc.value[0], bc.value[1]);
    if (bc.type == 1) {
        const Source c = src[j];
        double2 pin = make_double2(0.0, 0.0), qin = make_double2(0.0, 0.0);
        for (int64_t w = 0; w < nsrc; ++w) {
            double2 p, q;
            incident_value(srcs[w], c.c, c.n, k, hf, &p, &q);
            pin = cadd(pin, p);
            qin = cadd(qin, q);
        }
        pe[j] = csub(val, pin);
        const double2 q = csub(s, qin);
        // q / (i pf) as a complex division, zero when pf vanishes
        ve[j] = fabs(pf) > 1e-30 ? make_double2(q.y * pf / (pf * pf), -q.x * pf / (pf * pf)) : make_double2(0.0, 0.0);
    } else {
        pe[j] = s;
        ve[j] = bc.has_adm ? cadd(val, cmul(make_double2(bc.adm[0], bc.adm[1]), s)) : val;
    }
}

__global__ void sincos_probe_kernel(const double* x, int64_t n, double* s, double* c) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) sincos_red(x[t], &s[t], &c[t]);
}

}  // namespace

void upload_quadrature_tables(sbh_context* ctx) {
    double X[9][8] = {}, W[9][8] = {};
    for (int o = 1; o <= 8; ++o) gauss_legendre_rule(o, X[o], W[o]);
    SBH_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kGlX), X, sizeof(X)));
    SBH_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kGlW), W, sizeof(W)));
    (void)ctx;
}

// Calls launch(mode, variant) with the far loop's compile-time arguments.
template <typename Launch>
static void with_far_variant(int variant, int general, Launch&& launch) {
    auto mode = [&](auto var) {
        if (general)
            launch(std::integral_constant<int, 1>(), var);
        else
            launch(std::integral_constant<int, 0>(), var);
    };
    if (variant == FAR_SHORT)
        mode(std::integral_constant<int, FAR_SHORT>());
    else if (variant == FAR_LONG)
        mode(std::integral_constant<int, FAR_LONG>());
    else
        mode(std::integral_constant<int, FAR_GENERAL>());
}

// Near pairs per workgroup: 256 fill the lanes of its leaf passes best (8 leaves
// a pair on average, a partial pass per workgroup); fewer where that would
// leave less than two workgroups per CU.
static int near_pairs_per_block(int64_t npairs) {
    int per = 256;
    while (per > 32 && npairs / per < 512) per /= 2;
    return per;
}

void launch_assembly(sbh_workspace* ws, const sbh_physics& ph, sbh_c64 beta_c, sbh_system* sys) {
    injection_check(INJECT_LAUNCH);
    sbh_context* ctx = ws->ctx;
    const sbh_mesh* m = ws->mesh;
    const int64_t n = m->n;
    const double k = ph.wave_number;
    const double wavruim = ph.harmonic_factor * ph.wave_number;
    const double2 beta = make_double2(beta_c.re, beta_c.im);
    const double2 iwr = make_double2(0.0, ph.pressure_factor);
    if (n == 0) return;
    // The sin/cos argument reduction is valid for |k r| < 2^20.
    SBH_REQUIRE(std::fabs(k) * m->diameter < 5.0e5,
                "k * mesh diameter exceeds the supported phase range (5e5 rad)");
    if (ph.harmonic_factor != 1.0)
        throw Error(SBH_ERR_UNSUPPORTED, "only harmonic_factor = +1 (ACOUSTIC_CONVENTION) is supported");
    const int general = m->general ? 1 : 0;
    int rows_per_block = 16;
    while ((n + rows_per_block - 1) / rows_per_block > 65535) rows_per_block *= 2;
    dim3 grid((unsigned)((n + 255) / 256), (unsigned)((n + rows_per_block - 1) / rows_per_block));
    // row maxima for a low-precision copy of this system (only while one
    // exists), valid once every kernel below has run
    sys->rowmax_valid = false;
    const int64_t nbx = sys->rowmax_stride;
    const bool row_max = sys->lowp_copies.load() > 0 && rows_per_block <= FAR_MAX_ROWS && nbx == (int64_t)grid.x + 1 && sys->d_rowmax.ptr &&
                         ws->d_row_ptr.ptr && !sys->matrix_exposed;
    double* rm = row_max ? sys->d_rowmax.ptr : nullptr;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_FAR, &ev);
    with_far_variant(far_variant(k, m->panel_radius, beta.x), general, [&](auto mode, auto var) {
        hipLaunchKernelGGL((far_kernel<decltype(mode)::value, decltype(var)::value>), grid, dim3(256), 0, ctx->stream,
                           m->d_far.ptr, m->d_src.ptr, m->d_bc.ptr, n, sys->lda, rows_per_block, k, ph.tau, beta, iwr,
                           sys->d_A.ptr, ws->d_row_ptr.ptr, ws->d_pairs.ptr, rm, nbx);
    });
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_FAR, ev);
    if (ws->near_pairs > 0) {
        ctx->begin_timed(SBH_KERNEL_ASSEMBLE_NEAR, &ev);
        const int per = near_pairs_per_block(ws->near_pairs);
        with_far_variant(far_variant(k, m->panel_radius, beta.x), general, [&](auto mode, auto var) {
            hipLaunchKernelGGL((near_kernel<decltype(mode)::value, decltype(var)::value>),
                               dim3((unsigned)((ws->near_pairs + per - 1) / per)), dim3(256), 0, ctx->stream,
                               ws->d_pairs.ptr, ws->near_pairs, per, ws->d_leaves.ptr, m->d_far.ptr, m->d_src.ptr,
                               m->d_bc.ptr, sys->lda, k, ph.tau, beta, iwr, sys->d_A.ptr, rm, nbx);
        });
        SBH_HIP(hipGetLastError());
        ctx->end_timed(SBH_KERNEL_ASSEMBLE_NEAR, ev);
    }
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_SELF, &ev);
    hipLaunchKernelGGL(self_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, ctx->stream,
                       m->d_geom.ptr, m->d_src.ptr, m->d_bc.ptr, general, n, sys->lda, k, wavruim,
                       ph.tau, beta, iwr, sys->d_A.ptr, sys->d_rhs.ptr, rm, nbx);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_SELF, ev);
    sys->rowmax_valid = row_max;
    const int64_t ncols = (int64_t)m->nonzero_bc.size();
    if (ncols > 0) {
        ctx->begin_timed(SBH_KERNEL_RHS, &ev);
        hipLaunchKernelGGL(bc_rhs_kernel, dim3((unsigned)n), dim3(256), 0, ctx->stream,
                           m->d_nonzero_bc.ptr, ncols, ws->d_pairs.ptr, ws->d_row_ptr.ptr,
                           ws->d_leaves.ptr, m->d_geom.ptr, m->d_src.ptr, m->d_bc.ptr, k, wavruim,
                           ph.tau, beta, iwr, sys->d_rhs.ptr);
        SBH_HIP(hipGetLastError());
        ctx->end_timed(SBH_KERNEL_RHS, ev);
    }
}

void launch_source_rhs(sbh_context* ctx, const sbh_mesh* m, const sbh_physics& ph, sbh_c64 beta, double sign,
                       const IncidentSource* d_sources, int64_t nsources, double2* rhs, bool accumulate) {
    const int64_t n = m->n;
    if (n == 0) return;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_RHS, &ev);
    hipLaunchKernelGGL(source_rhs_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, m->d_src.ptr,
                       n, d_sources, nsources, ph.wave_number, ph.harmonic_factor, ph.tau,
                       make_double2(beta.re, beta.im), sign, accumulate ? 1 : 0, rhs);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_RHS, ev);
}

void launch_derivative_assembly(sbh_workspace* ws, const sbh_physics& ph, sbh_c64 beta, sbh_c64 beta_d,
                                double sign, double wavenumber_scale, double pf_derivative, double admittance_scale,
                                sbh_system* sys) {
    sbh_context* ctx = ws->ctx;
    const sbh_mesh* m = ws->mesh;
    const int64_t n = m->n;
    if (n == 0) return;
    SBH_REQUIRE(std::fabs(ph.wave_number) * m->diameter < 5.0e5,
                "k * mesh diameter exceeds the supported phase range (5e5 rad)");
    if (ph.harmonic_factor != 1.0)
        throw Error(SBH_ERR_UNSUPPORTED, "only harmonic_factor = +1 (ACOUSTIC_CONVENTION) is supported");
    DerivParams P;
    P.k = ph.wave_number;
    P.wavruim = ph.harmonic_factor * ph.wave_number;
    P.hf = ph.harmonic_factor;
    P.tau_r = ph.tau;
    P.sign = sign;
    P.ws = wavenumber_scale;
    P.adm_scale = admittance_scale;
    P.beta = make_double2(beta.re, beta.im);
    P.beta_d = make_double2(beta_d.re, beta_d.im);
    P.iwr = make_double2(0.0, ph.pressure_factor);
    P.iwr_d = make_double2(0.0, pf_derivative);
    const int general = m->general ? 1 : 0;
    sys->rowmax_valid = false;  // the matrix now holds a derivative
    int rows_per_block = 16;
    while ((n + rows_per_block - 1) / rows_per_block > 65535) rows_per_block *= 2;
    const dim3 grid((unsigned)((n + 255) / 256), (unsigned)((n + rows_per_block - 1) / rows_per_block));
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_FAR, &ev);
    const int variant = far_variant(P.k, m->panel_radius, beta.re != 0.0 ? beta.re : beta_d.re);
    with_far_variant(variant, general, [&](auto mode, auto var) {
        hipLaunchKernelGGL((far_deriv_kernel<decltype(mode)::value, decltype(var)::value>), grid, dim3(256), 0,
                           ctx->stream, m->d_far.ptr, m->d_src.ptr, m->d_bc.ptr, n, sys->lda, rows_per_block, P,
                           sys->d_A.ptr);
    });
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_FAR, ev);
    if (ws->near_pairs > 0) {
        ctx->begin_timed(SBH_KERNEL_ASSEMBLE_NEAR, &ev);
        const int per = near_pairs_per_block(ws->near_pairs);
        with_far_variant(variant, general, [&](auto mode, auto var) {
            hipLaunchKernelGGL((near_deriv_kernel<decltype(mode)::value, decltype(var)::value>),
                               dim3((unsigned)((ws->near_pairs + per - 1) / per)), dim3(256), 0, ctx->stream,
                               ws->d_pairs.ptr, ws->near_pairs, per, ws->d_leaves.ptr, m->d_far.ptr, m->d_src.ptr,
                               m->d_bc.ptr, sys->lda, P, sys->d_A.ptr);
        });
        SBH_HIP(hipGetLastError());
        ctx->end_timed(SBH_KERNEL_ASSEMBLE_NEAR, ev);
    }
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_SELF, &ev);
    hipLaunchKernelGGL(self_deriv_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, ctx->stream, m->d_geom.ptr,
                       m->d_src.ptr, m->d_bc.ptr, general, n, sys->lda, P, sys->d_A.ptr, sys->d_rhs.ptr);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_SELF, ev);
    const int64_t ncols = (int64_t)m->nonzero_bc.size();
    if (ncols > 0) {
        ctx->begin_timed(SBH_KERNEL_RHS, &ev);
        hipLaunchKernelGGL(bc_rhs_deriv_kernel, dim3((unsigned)n), dim3(256), 0, ctx->stream,
                           m->d_nonzero_bc.ptr, ncols, ws->d_pairs.ptr, ws->d_row_ptr.ptr, ws->d_leaves.ptr,
                           m->d_geom.ptr, m->d_src.ptr, m->d_bc.ptr, P, sys->d_rhs.ptr);
        SBH_HIP(hipGetLastError());
        ctx->end_timed(SBH_KERNEL_RHS, ev);
    }
}

void launch_incident_rhs(sbh_context* ctx, const sbh_mesh* m, const sbh_physics& ph, sbh_c64 beta,
                         double sign, const double* d_dirs, const double2* d_amps, int64_t num_rhs,
                         double2* d_rhs, bool accumulate) {
    const int64_t total = m->n * num_rhs;
    if (total == 0) return;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_RHS, &ev);
    hipLaunchKernelGGL(plane_wave_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       ctx->stream, m->d_src.ptr, m->n, d_dirs, d_amps, num_rhs, ph.wave_number,
                       ph.harmonic_factor, ph.tau, make_double2(beta.re, beta.im), sign,
                       accumulate ? 1 : 0, d_rhs);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_RHS, ev);
}

void launch_batch_assembly(sbh_context* ctx, const BatchAssemblyArgs& args, int grid) {
    if (args.nitems == 0) return;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_FAR, &ev);
    hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(2), 0, ctx->stream, args.counter);
    SBH_HIP(hipGetLastError());
    if (args.nfamilies > 0) {
        const int64_t nb = (args.family_max_n + 255) / 256;
        const int64_t rb = (args.family_max_n + FAMILY_ROWS - 1) / FAMILY_ROWS;
        SBH_REQUIRE(nb < 65536 && rb < 65536 && args.nfamilies < 65536, "frequency-family grid out of range");
        for (int c = 0; c < FAMILY_CLASSES; ++c) {
            const int fb = c ? args.family_class_end[c - 1] : 0, fe = args.family_class_end[c];
            if (fe == fb) continue;
            const dim3 grid((unsigned)nb, (unsigned)rb, (unsigned)(fe - fb));
            const FreqFamily* fams = args.families + fb;
            if (c == 0)
                hipLaunchKernelGGL(batch_far_family_kernel<16>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.far, args.src, args.A);
            else if (c == 1)
                hipLaunchKernelGGL(batch_far_family_kernel<8>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.far, args.src, args.A);
            else if (c == 2)
                hipLaunchKernelGGL(batch_far_family_kernel<4>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.far, args.src, args.A);
            else
                hipLaunchKernelGGL(batch_far_family_kernel<2>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.far, args.src, args.A);
            SBH_HIP(hipGetLastError());
        }
    }
    hipLaunchKernelGGL(batch_assemble_kernel<0>, dim3((unsigned)grid), dim3(256), 0, ctx->stream, args);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_FAR, ev);
    ctx->begin_timed(SBH_KERNEL_ASSEMBLE_NEAR, &ev);
    if (args.nfamilies > 0 && args.family_max_pairs > 0) {
        const int64_t per_block = 256 / NEAR_FAMILY_LANES;
        const int64_t nb = std::min<int64_t>((args.family_max_pairs + per_block - 1) / per_block, 16384);
        for (int c = 0; c < FAMILY_CLASSES; ++c) {
            const int fb = c ? args.family_class_end[c - 1] : 0, fe = args.family_class_end[c];
            if (fe == fb) continue;
            const dim3 grid((unsigned)nb, (unsigned)(fe - fb));
            const FreqFamily* fams = args.families + fb;
            if (c == 0)
                hipLaunchKernelGGL(batch_near_family_kernel<16>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.pairs, args.leaves, args.geom, args.src, args.A);
            else if (c == 1)
                hipLaunchKernelGGL(batch_near_family_kernel<8>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.pairs, args.leaves, args.geom, args.src, args.A);
            else if (c == 2)
                hipLaunchKernelGGL(batch_near_family_kernel<4>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.pairs, args.leaves, args.geom, args.src, args.A);
            else
                hipLaunchKernelGGL(batch_near_family_kernel<2>, grid, dim3(256), 0, ctx->stream, fams, args.inst,
                                   args.pairs, args.leaves, args.geom, args.src, args.A);
            SBH_HIP(hipGetLastError());
        }
    }
    hipLaunchKernelGGL(batch_assemble_kernel<1>, dim3((unsigned)grid), dim3(256), 0, ctx->stream, args);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_ASSEMBLE_NEAR, ev);
}

void launch_exact_apply(const sbh_operator* op, const double2* x, double2* y) {
    const sbh_workspace* ws = op->ws;
    const sbh_mesh* m = ws->mesh;
    sbh_context* ctx = op->ctx;
    const int64_t n = m->n;
    const sbh_physics& ph = op->physics;
    const double k = ph.wave_number;
    const double wavruim = ph.harmonic_factor * ph.wave_number;
    const double2 beta = op->beta;
    const double2 iwr = make_double2(0.0, ph.pressure_factor);
    const int general = m->general ? 1 : 0;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_MATVEC, &ev);
    const dim3 far_grid((unsigned)((n + EXACT_ROWS - 1) / EXACT_ROWS));
    const int per = near_pairs_per_block(ws->near_pairs);
    with_far_variant(far_variant(k, m->panel_radius, beta.x), general, [&](auto mode, auto var) {
        constexpr int MODE = decltype(mode)::value, VAR = decltype(var)::value;
        hipLaunchKernelGGL((exact_far_kernel<MODE, VAR>), far_grid, dim3(256), 0, ctx->stream, m->d_far.ptr,
                           m->d_src.ptr, m->d_bc.ptr, n, k, ph.tau, beta, iwr, x, op->d_far.ptr);
        SBH_HIP(hipGetLastError());
        if (ws->near_pairs > 0)
            hipLaunchKernelGGL((exact_near_kernel<MODE, VAR>), dim3((unsigned)((ws->near_pairs + per - 1) / per)),
                               dim3(256), 0, ctx->stream, ws->d_pairs.ptr, ws->near_pairs, per, ws->d_leaves.ptr,
                               m->d_far.ptr, m->d_src.ptr, m->d_bc.ptr, k, ph.tau, beta, iwr, x, op->d_near.ptr);
    });
    SBH_HIP(hipGetLastError());
    hipLaunchKernelGGL(exact_self_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, ctx->stream, m->d_geom.ptr,
                       m->d_src.ptr, m->d_bc.ptr, general, n, k, wavruim, ph.tau, beta, iwr, x, op->d_self.ptr);
    SBH_HIP(hipGetLastError());
    hipLaunchKernelGGL(exact_combine_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream,
                       op->d_far.ptr, op->d_near.ptr, ws->d_row_ptr.ptr, op->d_self.ptr, n, op->sign, y);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_MATVEC, ev);
}

void launch_field(sbh_context* ctx, const sbh_mesh* m, const sbh_physics& ph, const double2* sol, const double2* v,
                  const double* d_points, int64_t npts, const IncidentSource* d_sources, int64_t nsources,
                  double2* scattered, double2* incident, double2* total) {
    const int64_t n = m->n;
    if (npts == 0) return;
    const double k = ph.wave_number, hf = ph.harmonic_factor, pf = ph.pressure_factor;
    const double2* p = sol;
    WorkArray<double2> pe, ve;
    if (!v && m->general) {
        pe.allocate((size_t)n);
        ve.allocate((size_t)n);
        hipLaunchKernelGGL(field_cauchy_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream,
                           m->d_bc.ptr, m->d_src.ptr, sol, n, d_sources, nsources, k, hf, pf, pe.ptr, ve.ptr);
        SBH_HIP(hipGetLastError());
        p = pe.ptr;
        v = ve.ptr;
    }
    const int64_t row_blocks = (npts + FIELD_ROWS - 1) / FIELD_ROWS;
    SBH_REQUIRE(row_blocks < ((int64_t)1 << 31), "too many evaluation points");
    // Enough workgroups to fill the chip: split the panels when the points alone give few.
    const int64_t chunks = (n + 255) / 256;
    const int64_t slices = std::max<int64_t>(1, std::min<int64_t>({chunks, 2048 / row_blocks, 65535}));
    const int64_t per_slice = (chunks + slices - 1) / slices * 256;
    WorkArray<double2> part((size_t)(slices * npts));
    const dim3 grid((unsigned)row_blocks, (unsigned)slices);
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_FIELD, &ev);
    with_far_variant(far_variant(hf * k, m->panel_radius, 0.0), v ? 1 : 0, [&](auto has_v, auto var) {
        hipLaunchKernelGGL((field_kernel<decltype(has_v)::value, decltype(var)::value>), grid, dim3(256), 0,
                           ctx->stream, m->d_far.ptr, n, d_points, npts, p, v, hf * k, pf, per_slice, part.ptr);
    });
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_FIELD, ev);
    hipLaunchKernelGGL(field_finish_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, ctx->stream, part.ptr,
                       (int)slices, d_points, npts, d_sources, nsources, k, hf, scattered, incident, total);
    SBH_HIP(hipGetLastError());
    SBH_HIP(hipStreamSynchronize(ctx->stream));  // the temporaries are freed on return
}

__global__ void rsqrt_probe_kernel(const double* x, int64_t n, double* y) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) y[t] = rsqrt_nr(x[t]);
}

void launch_rsqrt_probe(sbh_context* ctx, const double* x, int64_t n, double* y) {
    if (n == 0) return;
    hipLaunchKernelGGL(rsqrt_probe_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, x, n, y);
    SBH_HIP(hipGetLastError());
}

void launch_sincos_probe(sbh_context* ctx, const double* x, int64_t n, double* s, double* c) {
    if (n == 0) return;
    hipLaunchKernelGGL(sincos_probe_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       ctx->stream, x, n, s, c);
    SBH_HIP(hipGetLastError());
}

}  // namespace sbh
