// adjbody.h -- per (beam, bin) body of the adjoint of the far-field amplitude
// (host + device, so the tests can run it on the CPU).
//
// Model.  For a triangular aperture with vertices v_l (global frame), centre
// c = mean(v_l), right-handed normal n = N / |N|, N = (v_1 - v_0) x (v_2 - v_0), the
// amplitude `diffraction` (diff_mod.f90:576-670) puts on a bin at x is
//     A = s (g I + h J) C T_phi,     s = e^{i k |x - c|} (i / lambda) F(q),
// where C is the amplitude matrix with the reference's anti-parallel sign
// (diff_mod.f90:561-571), T_phi = temp_rot1 (diff_mod.f90:646-650), J = [[0,1],[-1,0]],
// F(q) = int_T e^{i q.(u - c)} dA the aperture's form factor at q = k (prop - khat),
// khat = (x - c) / |x - c|, and g, h the two numbers of the Karczewski-Wolf matrix
// and the scattering-plane rotation, rot4 . diff_ampl = g I + h J (diff_mod.f90:
// 124-198, 630-643), written with the aperture frame e_z = -n, e_y = unit(e_z x prop),
// e_x = e_y x e_z (the frame get_rotation_matrix2 and rot2 build,
// diff_mod.f90:200-289, 533-547):
//     k_j = khat.e_j, sq = sqrt(1 - k_2^2), m = (e_y - k_2 khat) / sq,
//     evo = (khat x e_y) / sqrt(1 - k_2^2), hc = unit(inc x khat) (or the theta_i bin),
//     p = hc.m, qh = hc.evo, da = -(Kz sq + k_3 / sq) / 2, db = -k_1 k_2 / (2 sq),
//     g = p da + qh db, h = p db - qh da.
// This equals the reference's formula up to rounding (the split contour sum of
// contour_integral is the same F, +i F for the clockwise aperture frame).
//
// Adjoint.  Given Lam = dL/dA (as re/im pairs: dL = Re sum conj(Lam) dA), the body
// adds this bin's part of dL/dC and of the per-beam sums from which dL/dv_l follows
// (adj_finish):
//   * the form factor at fixed q: dF/dv_l = a_l F + q (a_l . grad_q F), a_l =
//     d|N|/dv_l / |N| (= the gradient of the barycentric coordinate l), so
//     sum over bins of Re(nu F) and of q Re(nu grad F) suffice;
//   * c through khat (q and the polarisation) and through the phase k |x - c|;
//   * the frame through e_z = -n.
// Per-edge phase terms are recomputed, never stored.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <vector>

#include "ffbody.h"
#include "records.h"
#include "trig.h"

namespace abt {

// Per-bin inputs of the adjoint: bin position, the theta_i bin of the same phi (forward
// fallback of hc), |x| and k|x|/(2 pi); Lam' = Lam T_phi^T (re/im, Fortran pair order).
struct AdjBin {
    double x, y, z, xt, yt, rad, kr_rev;
};

// Per-beam constants (from the prepared record).
struct AdjBeam {
    double c[3], cc;            // centre, |c|^2
    double ex[3], ey[3], ez[3]; // aperture frame
    double P[3], Kz;            // propagation vector, P.e_z
    double C[8];                // sigma * ampl
    double xl[3], yl[3];        // in-plane coordinates of v_l - c
    double xr[3], yr[3];        // the same over 2 pi (mixed body: phases in revolutions)
    double area;                // |N| / 2
    double qa2;                 // (aperture radius)^2: series branch when |q|^2 qa2 < SERIES_QA^2
    // FP64 body
    const double* r;            // the record, for what only rare bins need (FP64 adjoint)
    double tA;                  // 2 area / (lambda EXP_H^2)
    double Px, Py;              // P.e_x, P.e_y
    double tx[3], ty[3];        // in-plane coordinates of v_l - c in table steps times 1 / k
    double U[4], V[4];          // sigma * ampl in the eigenvectors of g I + h J: C1 + i C2, C1 - i C2 by column
    // FP32 copies for the mixed-precision body
    float fex[3], fey[3], fez[3], fP[3], fKz, fC[8];
    float fxl[3], fyl[3];
    float fso;                  // orientation sign of (xl, yl) for the edge form
};

struct AdjAcc {
    double GC[8];               // dL/dC (re/im pairs)
    double S0;                  // sum Re(nu F)
    double Qx[3], Qy[3];        // sum q Re(nu dF/dq_x), sum q Re(nu dF/dq_y)
    double cb[3];               // dL/dc through khat, the phase and the fallback hc
    double exb[3], eyb[3], ezb[3];
};

template <class Rec>
__host__ __device__ inline void adj_beam_from_record(Rec r, AdjBeam& B)
{
    for (int i = 0; i < 3; i++) {
        B.c[i] = r[R_COM + i];
        B.ex[i] = r[R_RR + i];
        B.ey[i] = r[R_RR + 3 + i];
        B.ez[i] = r[R_RR + 6 + i];
        B.P[i] = r[R_PROP0 + i];
        B.xl[i] = r[R_EX + i];
        B.yl[i] = r[R_EY + i];
        B.xr[i] = B.xl[i] * 0.15915494309189535;
        B.yr[i] = B.yl[i] * 0.15915494309189535;
    }
    B.cc = r[R_CC];
    B.Kz = B.P[0] * B.ez[0] + B.P[1] * B.ez[1] + B.P[2] * B.ez[2];
    B.Px = B.P[0] * B.ex[0] + B.P[1] * B.ex[1] + B.P[2] * B.ex[2];
    B.Py = B.P[0] * B.ey[0] + B.P[1] * B.ey[1] + B.P[2] * B.ey[2];
    for (int q = 0; q < 8; q++) B.C[q] = r[R_AMPL + q];
    for (int c = 0; c < 2; c++) {
        const double* C = B.C + 4 * c;
        B.U[2 * c] = C[0] - C[3];
        B.U[2 * c + 1] = C[1] + C[2];
        B.V[2 * c] = C[0] + C[3];
        B.V[2 * c + 1] = C[1] - C[2];
    }
    B.area = fabs(r[R_AREA]);
    B.r = (const double*)r;
    B.tA = 2.0 * B.area * r[R_IL] / (EXP_H * EXP_H);
    for (int i = 0; i < 3; i++) {
        B.tx[i] = r[R_TX + i];
        B.ty[i] = r[R_TY + i];
    }
    B.qa2 = r[R_AMAX] * r[R_AMAX];
    for (int i = 0; i < 3; i++) {
        B.fex[i] = (float)B.ex[i];
        B.fey[i] = (float)B.ey[i];
        B.fez[i] = (float)B.ez[i];
        B.fP[i] = (float)B.P[i];
        B.fxl[i] = (float)B.xl[i];
        B.fyl[i] = (float)B.yl[i];
    }
    B.fKz = (float)B.Kz;
    for (int q = 0; q < 8; q++) B.fC[q] = (float)B.C[q];
    const double a2 = (B.xl[1] - B.xl[0]) * (B.yl[2] - B.yl[0]) - (B.xl[2] - B.xl[0]) * (B.yl[1] - B.yl[0]);
    B.fso = a2 < 0.0 ? 1.0f : -1.0f;
}

// FP32 partial sums of the mixed body over a group of bins, added into AdjAcc
struct AdjAccF {
    float GC[8], S0, Qx[3], Qy[3], cb[3], exb[3], eyb[3], ezb[3];
};

__host__ __device__ inline void adj_zero_f(AdjAccF& a)
{
    for (int q = 0; q < 8; q++) a.GC[q] = 0.f;
    a.S0 = 0.f;
    for (int i = 0; i < 3; i++) {
        a.Qx[i] = a.Qy[i] = a.cb[i] = 0.f;
        a.exb[i] = a.eyb[i] = a.ezb[i] = 0.f;
    }
}

__host__ __device__ inline void adj_add(AdjAcc& a, const AdjAccF& f)
{
    for (int q = 0; q < 8; q++) a.GC[q] += (double)f.GC[q];
    a.S0 += (double)f.S0;
    for (int i = 0; i < 3; i++) {
        a.Qx[i] += (double)f.Qx[i];
        a.Qy[i] += (double)f.Qy[i];
        a.cb[i] += (double)f.cb[i];
        a.exb[i] += (double)f.exb[i];
        a.eyb[i] += (double)f.eyb[i];
        a.ezb[i] += (double)f.ezb[i];
    }
}

// bins per FP32 partial sum of the mixed adjoint
constexpr int ADJ_GROUP = 8;

__host__ __device__ inline void adj_zero(AdjAcc& a)
{
    for (int q = 0; q < 8; q++) a.GC[q] = 0.0;
    a.S0 = 0.0;
    for (int i = 0; i < 3; i++) {
        a.Qx[i] = a.Qy[i] = a.cb[i] = 0.0;
        a.exb[i] = a.eyb[i] = a.ezb[i] = 0.0;
    }
}

// sin(x)/x
__host__ __device__ __forceinline__ double sinc64(double x)
{
    const double z = x * x;
    if (fabs(x) < 0.5)
        return 1.0 + z * (-1.0 / 6 + z * (1.0 / 120 + z * (-1.0 / 5040 + z * (1.0 / 362880 + z * (-1.0 / 39916800)))));
    double s, c;
    sincos_f64(x, &s, &c);
    return s / x;
}

// F(q) and grad_q F of the triangle (in-plane coordinates xl, yl about the centre, either
// orientation) by the series about q = (qx, qy) = 0 (rad/um), for |q| a < SERIES_QA: complete
// homogeneous symmetric polynomials of the vertex phases and their derivatives.
__host__ __device__ inline void tri_series_grad(const double* __restrict__ xl, const double* __restrict__ yl,
                                                double area, double qx, double qy, double F[2], double Gx[2],
                                                double Gy[2])
{
    double al[3];
    for (int l = 0; l < 3; l++) al[l] = qx * xl[l] + qy * yl[l];
    const double e1 = al[0] + al[1] + al[2];
    const double e2 = al[0] * al[1] + al[1] * al[2] + al[2] * al[0];
    const double e3 = al[0] * al[1] * al[2];
    double hm3 = 0.0, hm2 = 0.0, hm1 = 1.0;          // h_{n-3}, h_{n-2}, h_{n-1} at n = 1
    double d[3] = {0.0, 0.0, 0.0};                    // h_{n-1}(al_l, al) at n = 0
    double f[2] = {0.5, 0.0};                         // n = 0 term: h_0 / 2!
    double g[2][3] = {{0, 0, 0}, {0, 0, 0}};
    double inv = 0.5, sign = 1.0;
    // pairs (odd, even) of n: i^n has the sign + - - + by pairs on f[1], f[0]
    for (int n = 1; n <= 23; n += 2) {
        for (int h = 0; h < 2; h++) {
            // d^{(l)}_{n-1} = h_{n-1} + al_l d^{(l)}_{n-2}
            for (int l = 0; l < 3; l++) d[l] = hm1 + al[l] * d[l];
            const double hn = e1 * hm1 - e2 * hm2 + e3 * hm3;
            inv *= rcp_cr((double)(n + h + 2));
            if (h == 1) sign = -sign;
            const double t = sign * inv;
            f[1 - h] += hn * t;
            for (int l = 0; l < 3; l++) g[1 - h][l] += d[l] * t;
            hm3 = hm2; hm2 = hm1; hm1 = hn;
        }
    }
    const double A2 = 2.0 * area;
    for (int c = 0; c < 2; c++) {
        F[c] = A2 * f[c];
        Gx[c] = A2 * (g[c][0] * xl[0] + g[c][1] * xl[1] + g[c][2] * xl[2]);
        Gy[c] = A2 * (g[c][0] * yl[0] + g[c][1] * yl[1] + g[c][2] * yl[2]);
    }
}

// F(q): the series, or the edge form F = (i/|q|^2) sum_j c_j sinc(q.e_j/2) e^{i q.m_j}.
__host__ __device__ inline void tri_ff(const AdjBeam& B, double qx, double qy, double F[2])
{
    const double q2 = qx * qx + qy * qy;
    if (q2 * B.qa2 < 2.25) {
        double Gx[2], Gy[2];
        tri_series_grad(B.xl, B.yl, B.area, qx, qy, F, Gx, Gy);
        return;
    }
    // orientation of (xl, yl): the edge form is for counter-clockwise order
    const double a2 = (B.xl[1] - B.xl[0]) * (B.yl[2] - B.yl[0]) - (B.xl[2] - B.xl[0]) * (B.yl[1] - B.yl[0]);
    const double so = a2 < 0.0 ? 1.0 : -1.0;
    double sr = 0, si = 0;
    for (int j = 0; j < 3; j++) {
        const int jn = j == 2 ? 0 : j + 1;
        const double ex = B.xl[jn] - B.xl[j], ey = B.yl[jn] - B.yl[j];
        double es, ec;
        sincos_f64(qx * (0.5 * (B.xl[j] + B.xl[jn])) + qy * (0.5 * (B.yl[j] + B.yl[jn])), &es, &ec);
        const double t = so * (qx * ey - qy * ex) * sinc64(0.5 * (qx * ex + qy * ey));
        sr += t * ec;
        si += t * es;
    }
    const double iq2 = 1.0 / q2;
    F[0] = -si * iq2;
    F[1] = sr * iq2;
}

__host__ __device__ __forceinline__ double dot3(const double* a, const double* b)
{
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

__host__ __device__ __forceinline__ void cross3(const double* a, const double* b, double* o)
{
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// Per-bin inputs of the FP64 body: direction and 1 / |x|, the theta_i bin of the same phi
// (forward fallback of hc), and k |x| in exponential-table steps, less whole turns.  x: the position.
struct AdjFarBin {
    FarBin f;
    double xt, yt, kr;
    const double* x;
};

__host__ __device__ __forceinline__ AdjFarBin adj_far_bin(const AdjBin& b)
{
    const double ir = 1.0 / b.rad;
    return {{b.x * ir, b.y * ir, b.z * ir, ir}, b.xt, b.yt, (2 * ETAB_N) * (b.kr_rev - rint(b.kr_rev)), &b.x};
}

// Sums of the FP64 body.  GU, GV: the amplitude gradient in the eigenvectors of g I + h J (below);
// Kzb: dL/dKz, which enters e_z through K_z = P.e_z.
struct AdjSum {
    double GU[4], GV[4], S0, Kzb;
    double Qx[3], Qy[3], cb[3], exb[3], eyb[3], ezb[3];
};

__host__ __device__ inline void adj_zero_sum(AdjSum& a)
{
    for (int q = 0; q < 4; q++) a.GU[q] = a.GV[q] = 0.0;
    a.S0 = a.Kzb = 0.0;
    for (int i = 0; i < 3; i++) a.Qx[i] = a.Qy[i] = a.cb[i] = a.exb[i] = a.eyb[i] = a.ezb[i] = 0.0;
}

// adds the FP64 body's sums to the accumulators that adj_finish reads
__host__ __device__ inline void adj_add_sum(const AdjBeam& B, const AdjSum& s, AdjAcc& a)
{
    for (int c = 0; c < 2; c++) {
        // G1 = GU + GV, G2 = -i (GU - GV)
        a.GC[4 * c] += s.GU[2 * c] + s.GV[2 * c];
        a.GC[4 * c + 1] += s.GU[2 * c + 1] + s.GV[2 * c + 1];
        a.GC[4 * c + 2] += s.GU[2 * c + 1] - s.GV[2 * c + 1];
        a.GC[4 * c + 3] += s.GV[2 * c] - s.GU[2 * c];
    }
    a.S0 += s.S0;
    for (int i = 0; i < 3; i++) {
        a.Qx[i] += s.Qx[i];
        a.Qy[i] += s.Qy[i];
        a.cb[i] += s.cb[i];
        a.exb[i] += s.exb[i];
        a.eyb[i] += s.eyb[i];
        a.ezb[i] += fma(s.Kzb, B.P[i], s.ezb[i]);
    }
}

// Lam' (re/im, Fortran pair order) in the eigenvectors of g I + h J, halved:
// (L1 + i L2) / 2 of columns 1, 2, then (L1 - i L2) / 2.
__host__ __device__ __forceinline__ void adj_lam_split(const double* L, double* o)
{
    for (int c = 0; c < 2; c++) {
        const double l1r = 0.5 * L[4 * c], l1i = 0.5 * L[4 * c + 1], l2r = 0.5 * L[4 * c + 2], l2i = 0.5 * L[4 * c + 3];
        o[2 * c] = l1r - l2i;
        o[2 * c + 1] = l1i + l2r;
        o[4 + 2 * c] = l1r + l2i;
        o[4 + 2 * c + 1] = l1i - l2r;
    }
}

// One edge of the form factor from the full vertex exponentials W (far-field phase included) of its
// ends: D = sinc(K/2) e^{i (alpha_0 + alpha_1)/2} = (W1 - W0) / (i K) and its derivatives by
// alpha_0 and alpha_1, K = alpha_1 - alpha_0 in rad; series of the product form for |K| < 1.
__host__ __device__ __forceinline__ void edge_grad64(double W0r, double W0i, double W1r, double W1i, double K,
                                                     double D[2], double D0[2], double D1[2])
{
    const double x = 0.5 * K;
    if (fabs(x) < 0.5) {
        const double z = x * x;
        const double S = 1.0 + z * (-1.0 / 6 + z * (1.0 / 120 + z * (-1.0 / 5040 + z * (1.0 / 362880 + z * (-1.0 / 39916800)))));
        const double hS = 0.5 * x * (-1.0 / 3 + z * (1.0 / 30 + z * (-1.0 / 840 + z * (1.0 / 45360 + z * (-1.0 / 3991680 + z * (1.0 / 518918400))))));
        double s, c;
        sincos_f64(x, &s, &c);
        const double mr = W0r * c - W0i * s, mi = W0r * s + W0i * c;   // e^{i (alpha_0 + alpha_1)/2}
        D[0] = S * mr;
        D[1] = S * mi;
        D0[0] = -0.5 * D[1] - hS * mr;
        D0[1] = 0.5 * D[0] - hS * mi;
        D1[0] = -0.5 * D[1] + hS * mr;
        D1[1] = 0.5 * D[0] + hS * mi;
    } else {
        const double iK = rcp_cr(K);
        D[0] = (W1i - W0i) * iK;
        D[1] = (W0r - W1r) * iK;
        D0[0] = (D[0] - W0r) * iK;
        D0[1] = (D[1] - W0i) * iK;
        D1[0] = (W1r - D[0]) * iK;
        D1[1] = (W1i - D[1]) * iK;
    }
}

// F e^{i k |x - c|} / lambda and its derivatives by (q_x, q_y) / k, for the bins where the one
// denominator of adj_bin_far does not hold: series about q = 0, or the edge form.
__host__ __device__ inline void tri_ff_grad_other(const double* __restrict__ r, const TriPhase& w, double qx, double qy, double kd,
                                                  const double* __restrict__ tab, double k, double F[2], double Gx[2],
                                                  double Gy[2])
{
    const double* xl = r + R_EX;
    const double* yl = r + R_EY;
    const double il = r[R_IL];
    double sc = k * il;
    if (fma(qx, qx, qy * qy) * (r[R_AMAX] * r[R_AMAX]) < 2.25) {
        double f[2], gx[2], gy[2], c, s;
        tri_series_grad(xl, yl, fabs(r[R_AREA]), qx, qy, f, gx, gy);
        expi_step64(kd, tab, &c, &s);
        F[0] = il * (c * f[0] - s * f[1]);
        F[1] = il * (c * f[1] + s * f[0]);
        c *= sc;
        s *= sc;
        Gx[0] = c * gx[0] - s * gx[1];
        Gx[1] = c * gx[1] + s * gx[0];
        Gy[0] = c * gy[0] - s * gy[1];
        Gy[1] = c * gy[1] + s * gy[0];
        return;
    }
    // F = (i / |q|^2) sum_j c_j D_j for counter-clockwise order
    const double a2 = (xl[1] - xl[0]) * (yl[2] - yl[0]) - (xl[2] - xl[0]) * (yl[1] - yl[0]);
    const double so = a2 < 0.0 ? 1.0 : -1.0;
    const double K[3] = {EXP_H * w.d0, EXP_H * w.d1, EXP_H * w.d2};
    double sr = 0, si = 0, gxr = 0, gxi = 0, gyr = 0, gyi = 0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const int jn = j == 2 ? 0 : j + 1;
        double D[2], D0[2], D1[2];
        edge_grad64(w.Wr[j], w.Wi[j], w.Wr[jn], w.Wi[jn], K[j], D, D0, D1);
        const double ex = so * (xl[jn] - xl[j]), ey = so * (yl[jn] - yl[j]);
        const double cj = qx * ey - qy * ex;
        sr += cj * D[0];
        si += cj * D[1];
        gxr += ey * D[0] + cj * (D0[0] * xl[j] + D1[0] * xl[jn]);
        gxi += ey * D[1] + cj * (D0[1] * xl[j] + D1[1] * xl[jn]);
        gyr += -ex * D[0] + cj * (D0[0] * yl[j] + D1[0] * yl[jn]);
        gyi += -ex * D[1] + cj * (D0[1] * yl[j] + D1[1] * yl[jn]);
    }
    const double iq2 = rcp_cr(fma(qx, qx, qy * qy)), tx = 2.0 * qx * iq2, ty = 2.0 * qy * iq2;
    sc *= iq2;
    F[0] = -si * iq2 * il;
    F[1] = sr * iq2 * il;
    Gx[0] = -gxi * sc - k * tx * F[0];
    Gx[1] = gxr * sc - k * tx * F[1];
    Gy[0] = -gyi * sc - k * ty * F[0];
    Gy[1] = gyr * sc - k * ty * F[1];
}

// The polarisation numbers g, h of one beam and bin and, for gg = dL/dg and gh = dL/dh, the adjoints
// of what they are made of: the three k_j, K_z, e_y (less its k_2 part), khat beyond the k_j, and
// in the forward fallback the centre.
struct AdjPol {
    double g, h, k1b, k2b, k3b, Kzb;
    double eyb[3], kb[3], cb0, cb1;
};

// Away from the clamp and the forward fallback, hc = unit(inc x khat) is normal to khat, so
// g = D (P0 A + Q0 B), h = D (P0 B - Q0 A) with D = 1 / (|inc x khat| (1 - k_2^2)), P0 = e_y . (kh_y, -kh_x, 0),
// Q0 = e_y . ((inc.khat) khat - inc), A = -(K_z (1 - k_2^2) + k_3) / 2, B = -k_1 k_2 / 2.
// is2 = 1 / s2, s2 = 1 - k_2^2.  The radial part of kb is left out where it is free: only the part of kb
// normal to khat is used.
__host__ __device__ __forceinline__ AdjPol adj_pol_fast(const AdjBeam& B, const FarGeom& u, double k1, double k2,
                                                        double k3, double s2, double is2, double gg, double gh)
{
    AdjPol o;
    const double P0 = fma(B.ey[0], u.uy, -B.ey[1] * u.ux);
    const double Q0 = fma(-u.uz, k2, B.ey[2]);
    const double rh = rsq64_3(fma(u.ux, u.ux, u.uy * u.uy));
    const double D = rh * is2;
    const double A = -0.5 * fma(B.Kz, s2, k3), Bq = -0.5 * k1 * k2;
    const double DA = D * A, DB = D * Bq;
    o.g = fma(P0, DA, Q0 * DB);
    o.h = fma(P0, DB, -Q0 * DA);
    const double Pb = fma(gg, DA, gh * DB), Qb = fma(gg, DB, -gh * DA);
    const double hD = -0.5 * D;
    const double Ab = hD * fma(gg, P0, -gh * Q0);          // -dL/dA / 2
    const double Bb = hD * fma(gg, Q0, gh * P0);           // -dL/dB / 2
    const double w = fma(gg, o.g, gh * o.h);               // D dL/dD
    const double rw = w * (rh * rh);
    o.Kzb = s2 * Ab;
    o.k3b = Ab;
    o.k1b = k2 * Bb;
    o.k2b = fma(k2, 2.0 * fma(w, is2, -B.Kz * Ab), fma(k1, Bb, -u.uz * Qb));
    o.kb[0] = fma(-rw, u.ux, -B.ey[1] * Pb);
    o.kb[1] = fma(-rw, u.uy, B.ey[0] * Pb);
    o.kb[2] = -k2 * Qb;
    o.eyb[0] = u.uy * Pb;
    o.eyb[1] = -u.ux * Pb;
    o.eyb[2] = Qb;
    o.cb0 = o.cb1 = 0.0;
    return o;
}

// Within the clamp 1 - k_2^2 is 2e-6 and less, so its rounding (1e-16) shows in p and qh; there it is formed
// from the position in the plain manner, as the forward model forms it.
__host__ __device__ inline AdjPol adj_pol_other(const AdjBeam& B, const FarGeom& u, const AdjFarBin& bn, double k1,
                                                double k2, double k3, bool clamp, bool fb, double gg, double gh)
{
    AdjPol o;
    const double kh[3] = {u.ux, u.uy, u.uz};
    const double k2c = clamp ? copysign(K2CLAMP, k2) : k2;
    const double sq = sqrt(1.0 - k2c * k2c), isq = 1.0 / sq;
    double s13q = fma(k1, k1, k3 * k3);                // 1 - k_2^2
    if (clamp) {
        const double d[3] = {bn.x[0] - B.c[0], bn.x[1] - B.c[1], bn.x[2] - B.c[2]};
        const double ir = 1.0 / sqrt(dot3(d, d));
        const double w[3] = {d[0] * ir, d[1] * ir, d[2] * ir};
        const double w2 = dot3(w, B.ey);
        s13q = 1.0 - w2 * w2;
    }
    const double is13 = 1.0 / sqrt(s13q);
    const double hx = fb ? bn.yt - B.c[1] : kh[1], hy = fb ? B.c[0] - bn.xt : -kh[0];
    const double inh = 1.0 / sqrt(hx * hx + hy * hy);
    const double hc[3] = {hx * inh, hy * inh, 0.0};
    double m[3], e[3], t[3];
    cross3(kh, B.ey, e);
    for (int i = 0; i < 3; i++) {
        m[i] = (B.ey[i] - k2c * kh[i]) * isq;
        e[i] *= is13;
    }
    const double p = dot3(hc, m), qh = dot3(hc, e);
    const double da = -0.5 * (B.Kz * sq + k3 * isq), db = -0.5 * k1 * k2c * isq;
    o.g = p * da + qh * db;
    o.h = p * db - qh * da;
    const double pb = gg * da + gh * db, qb = gg * db - gh * da;
    const double dab = gg * p - gh * qh, dbb = gg * qh + gh * p;
    o.Kzb = -0.5 * sq * dab;
    o.k3b = -0.5 * dab * isq;
    o.k1b = -0.5 * k2c * isq * dbb;
    const double mb[3] = {pb * hc[0], pb * hc[1], 0.0};
    const double ub[3] = {qb * hc[0] * is13, qb * hc[1] * is13, 0.0};
    const double sqb = -0.5 * (B.Kz - k3 * isq * isq) * dab + 0.5 * k1 * k2c * isq * isq * dbb - dot3(mb, m) * isq;
    const double k2cb = -0.5 * k1 * isq * dbb - dot3(mb, kh) * isq - k2c * isq * sqb;
    o.k2b = k2 * is13 * is13 * qb * qh;
    if (!clamp) o.k2b += k2cb;
    cross3(ub, kh, t);
    for (int i = 0; i < 3; i++) o.eyb[i] = mb[i] * isq + t[i];
    cross3(B.ey, ub, t);
    for (int i = 0; i < 3; i++) o.kb[i] = t[i] - k2c * isq * mb[i];
    // hc = hv / |hv|, hv = inc x khat (or inc x (x_t - c)); d/dy (inc x y).hvb = y.(hvb x inc)
    const double hcb0 = pb * m[0] + qb * e[0], hcb1 = pb * m[1] + qb * e[1];
    const double hdot = hcb0 * hc[0] + hcb1 * hc[1];
    const double tx = -(hcb1 - hdot * hc[1]) * inh, ty = (hcb0 - hdot * hc[0]) * inh;   // hvb x (0,0,-1)
    o.cb0 = fb ? -tx : 0.0;
    o.cb1 = fb ? -ty : 0.0;
    o.kb[0] += fb ? 0.0 : tx;
    o.kb[1] += fb ? 0.0 : ty;
    return o;
}

// One denominator for F and its gradient (adj_bin_far), d = d0 d1 d2 in table steps.  The exponentials'
// rounding (1.7e-16) enters dF / (2 A dalpha) as ~1.7e-16 max |K| / (|K0 K1 K2| min |K|), K_j = EXP_H d_j: at most
// 1.7e-13 of the 1/6 it has at q = 0 under the condition (min |K| of an edge seen at 100 rad across: 3e-3 rad).
__host__ __device__ __forceinline__ bool one_denominator_grad(const TriPhase& w, double d)
{
    const double a = fabs(w.d0), b = fabs(w.d1), c = fabs(w.d2);
    // strict: q = 0 has every d_j = 0.  The largest is half the sum, d0 + d1 + d2 = 0.
    return fabs(d) * fmin(a, fmin(b, c)) > (0.5e-3 / (EXP_H * EXP_H * EXP_H)) * (a + b + c);
}

// One (beam, bin) of the FP64 adjoint.  lam: Lam' = Lam T_phi^T from adj_lam_split; far: the beam's centre is
// within the far geometry's limit; tab: the exponential table; kt: its steps per um.
//
// Bound by FP64 VALU issue, as the forward body (ffbody.h), whose means it uses: the far geometry in
// series, phases in table steps, three vertex exponentials W_l = e^{i (alpha_l + k |x - c|)} in place of
// twelve trigonometric pairs, and, away from the edges' nulls and the clamp,
//   F = 2 A N / (K0 K1 K2), N = W0 K1 + W1 K2 + W2 K0, K_j = alpha_{j+1} - alpha_j,
// whose derivatives are taken as real numbers, rho_l = Re(nu dF/dalpha_l): with u + i v = nu f W (f N = F)
//   rho_0 = u_1 - u_2 - K_1 v_0 - Re(nu F) (1/K_2 - 1/K_0), and cyclic,
// from which q_x and q_y gather sum_l rho_l x_l, rho_l y_l.  The amplitude side works in the
// eigenvectors of g I + h J, U = C1 + i C2 (eigenvalue g - i h) and V = C1 - i C2 (g + i h): half the products.
// 396 instructions a beam and bin where six edge terms, each with its own trigonometry, took 1634: 5 orientations
// of the rough column (209 blocks of 64 beams) x 16,290 bins 15.2 -> 5.2 ms, 3.3 ms with finer chunks of bins,
// 3.1 ms with each bin's inputs loaded a bin ahead (k_adjoint64); the issue rate alone is 2.4 ms, the rest the last
// round of waves and waits that two waves per SIMD leave open.
__host__ __device__ __forceinline__ void adj_bin_far(const AdjBeam& B, const AdjFarBin& bn,
                                                     const double* __restrict__ lam, bool far,
                                                     const double* __restrict__ tab, double k, double kt,
                                                     AdjSum& acc)
{
    const FarGeom u = far_geometry(B.c, B.cc, kt, bn.f, far);
    const double kd = u.kd + bn.kr;
    const double k1 = fma(u.ux, B.ex[0], fma(u.uy, B.ex[1], u.uz * B.ex[2]));
    const double k2 = fma(u.ux, B.ey[0], fma(u.uy, B.ey[1], u.uz * B.ey[2]));
    const double k3 = fma(u.ux, B.ez[0], fma(u.uy, B.ez[1], u.uz * B.ez[2]));
    const double q1 = B.Px - k1, q2 = B.Py - k2;              // q / k in the aperture plane
    const TriPhase w = tri_phases_of(B.tx, B.ty, q1, q2, kd, tab);
    const double d12 = w.d1 * w.d2, d = w.d0 * d12;
    const bool one = one_denominator_grad(w, d);
    const bool clamp = fabs(k2) > K2CLAMP, fb = !(fabs(u.uz) < FWD_DOT);
    const bool fast = !clamp && !fb;
    const double s2 = fma(k1, k1, k3 * k3);                   // 1 - k_2^2
    double id, is2;
    if (one && fast) {
        const double r = rcp_cr(s2 * d);
        id = r * s2;
        is2 = r * d;
    } else {
        id = rcp_cr(d);
        is2 = rcp_cr(s2);
    }
    // F e^{i k |x - c|} / lambda
    double F[2], Gx[2], Gy[2];
    const double f = B.tA * id;
    if (one) {
        F[0] = f * fma(w.Wr[0], w.d1, fma(w.Wr[1], w.d2, w.Wr[2] * w.d0));
        F[1] = f * fma(w.Wi[0], w.d1, fma(w.Wi[1], w.d2, w.Wi[2] * w.d0));
        Gx[0] = Gx[1] = Gy[0] = Gy[1] = 0.0;
    } else {
        tri_ff_grad_other(B.r, w, k * q1, k * q2, kd, tab, k, F, Gx, Gy);
    }
    const double sr = -F[1], si = F[0];                       // s = i F
    // <Lam', U> and <Lam', V> over the columns; z1 = <Lam', C> = zu + zv, z2 = <Lam', J C> = -i (zu - zv)
    double zur = 0, zui = 0, zvr = 0, zvi = 0;
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
        zur = fma(lam[c], B.U[c], fma(lam[c + 1], B.U[c + 1], zur));
        zui = fma(lam[c], B.U[c + 1], fma(-lam[c + 1], B.U[c], zui));
        zvr = fma(lam[4 + c], B.V[c], fma(lam[5 + c], B.V[c + 1], zvr));
        zvi = fma(lam[4 + c], B.V[c + 1], fma(-lam[5 + c], B.V[c], zvi));
    }
    const double z1r = zur + zvr, z1i = zui + zvi, z2r = zui - zvi, z2i = zvr - zur;
    const double gg = fma(sr, z1r, -si * z1i), gh = fma(sr, z2r, -si * z2i);
    const AdjPol o = fast ? adj_pol_fast(B, u, k1, k2, k3, s2, is2, gg, gh)
                          : adj_pol_other(B, u, bn, k1, k2, k3, clamp, fb, gg, gh);
    // dL/dC = conj(s) (g I - h J) Lam'
    {
        const double ur = fma(sr, o.g, si * o.h), ui = fma(si, o.g, -sr * o.h);   // s (g - i h)
        const double vr = fma(sr, o.g, -si * o.h), vi = fma(si, o.g, sr * o.h);   // s (g + i h)
#pragma unroll
        for (int c = 0; c < 4; c += 2) {
            acc.GU[c] = fma(ur, lam[c], fma(ui, lam[c + 1], acc.GU[c]));
            acc.GU[c + 1] = fma(ur, lam[c + 1], fma(-ui, lam[c], acc.GU[c + 1]));
            acc.GV[c] = fma(vr, lam[4 + c], fma(vi, lam[5 + c], acc.GV[c]));
            acc.GV[c + 1] = fma(vr, lam[5 + c], fma(-vi, lam[4 + c], acc.GV[c + 1]));
        }
    }
    // nu = i (g z1 + h z2): nu F = its part of dL;  Rx = Re(nu dF/d(q_x / k)) = k Re(nu dF/dq_x)
    const double nur = -fma(o.g, z1i, o.h * z2i), nui = fma(o.g, z1r, o.h * z2r);
    double S, ph, Rx, Ry;
    if (one) {
        const double ar = nur * f, ai = nui * f, br = EXP_H * ar, bi = EXP_H * ai;
        double U[3], V[3];
#pragma unroll
        for (int l = 0; l < 3; l++) {
            U[l] = fma(ar, w.Wr[l], -ai * w.Wi[l]);
            V[l] = fma(br, w.Wi[l], bi * w.Wr[l]);
        }
        const double V0 = w.d1 * V[0], V1 = w.d2 * V[1], V2 = w.d0 * V[2];
        S = fma(U[0], w.d1, fma(U[1], w.d2, U[2] * w.d0));
        ph = (k / EXP_H) * (V0 + V1 + V2);
        const double Si = S * id;
        const double S0 = Si * d12, S1 = Si * (w.d2 * w.d0), S2 = Si * (w.d0 * w.d1);   // S / d_j
        const double r0 = (U[1] - U[2]) - V0 + (S0 - S2);
        const double r1 = (U[2] - U[0]) - V1 + (S1 - S0);
        const double r2 = (U[0] - U[1]) - V2 + (S2 - S1);
        Rx = fma(r0, B.tx[0], fma(r1, B.tx[1], r2 * B.tx[2]));
        Ry = fma(r0, B.ty[0], fma(r1, B.ty[1], r2 * B.ty[2]));
    } else {
        S = fma(nur, F[0], -nui * F[1]);
        ph = k * fma(nur, F[1], nui * F[0]);
        Rx = fma(nur, Gx[0], -nui * Gx[1]);
        Ry = fma(nur, Gy[0], -nui * Gy[1]);
    }
    acc.S0 += S;
    acc.Kzb += o.Kzb;
    const double kh[3] = {u.ux, u.uy, u.uz};
    const double b1 = o.k1b - Rx, b2 = o.k2b - Ry;            // q = k (P - khat) and the polarisation
    double kb[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double qk = B.P[i] - kh[i];
        acc.Qx[i] = fma(qk, Rx, acc.Qx[i]);
        acc.Qy[i] = fma(qk, Ry, acc.Qy[i]);
        kb[i] = fma(b1, B.ex[i], fma(b2, B.ey[i], fma(o.k3b, B.ez[i], o.kb[i])));
        acc.exb[i] = fma(o.k1b, kh[i], acc.exb[i]);
        acc.eyb[i] = fma(o.k2b, kh[i], acc.eyb[i] + o.eyb[i]);
        acc.ezb[i] = fma(o.k3b, kh[i], acc.ezb[i]);
    }
    // khat = d / rho, d = x - c:  dc = -(I - khat khat^T) kb / rho;  phase: k Im(nu F) khat
    const double kk = fma(kb[0], kh[0], fma(kb[1], kh[1], kb[2] * kh[2]));
    const double t = fma(kk, u.id, ph);
#pragma unroll
    for (int i = 0; i < 3; i++) acc.cb[i] = fma(t, kh[i], fma(-kb[i], u.id, acc.cb[i]));
    acc.cb[0] += o.cb0;
    acc.cb[1] += o.cb1;
}

// One (beam, bin) from plain inputs, on the host.  lam: Lam' = Lam T_phi^T (8 doubles).
inline void adj_bin_fp64(const AdjBeam& B, const AdjBin& bn, const double* __restrict__ lam, double waveno,
                         double lambda, AdjAcc& acc)
{
    static const std::vector<double> tab = [] {
        std::vector<double> t(ETAB_GRID);
        fill_exp_table(t.data());
        return t;
    }();
    (void)lambda;
    double ls[8];
    adj_lam_split(lam, ls);
    AdjSum s;
    adj_zero_sum(s);
    adj_bin_far(B, adj_far_bin(bn), ls, B.cc <= far_limit(waveno / 6.283185307179586, bn.rad), tab.data(), waveno,
                B.r[R_KT], s);
    adj_add_sum(B, s, acc);
}

// sin(x)/x and its derivative for |x| < 0.5 (FP32 series)
__host__ __device__ __forceinline__ float sinc_ser(float x)
{
    const float z = x * x;
    return fmaf(z, fmaf(z, fmaf(z, -1.98412698e-4f, 8.33333333e-3f), -0.166666667f), 1.0f);
}
__host__ __device__ __forceinline__ float dsinc_ser(float x)
{
    const float z = x * x;
    return x * fmaf(z, fmaf(z, fmaf(z, 2.20458554e-5f, -1.19047619e-3f), 3.33333333e-2f), -0.333333333f);
}

// Forward of the model in FP64 (the function the adjoint differentiates): adds
// s' (g I + h J) C to acc (re/im, Fortran pair order), s' = e^{i k (|x - c| - |x|)}
// (i / lambda) F with the phase formed without cancellation; the caller applies the
// per-bin e^{i k |x|} and T_phi after the beam sum (model_finish).  Agrees with the
// reference's formula to rounding and is smooth to ~1e-15, so finite differences
// with steps of 1e-4 um resolve its derivatives.
__host__ __device__ inline void model_bin_fp64(const AdjBeam& B, double x, double y, double z, double xt,
                                               double yt, double rad, double waveno, double lambda,
                                               double acc[8])
{
    const double k = waveno;
    const double d[3] = {x - B.c[0], y - B.c[1], z - B.c[2]};
    const double rho = sqrt(dot3(d, d));
    const double kh[3] = {d[0] / rho, d[1] / rho, d[2] / rho};
    const double rc = x * B.c[0] + y * B.c[1] + z * B.c[2];
    const double drho = (B.cc - 2.0 * rc) / (rho + rad);
    double Es, Ec;
    sincos_f64(k * drho, &Es, &Ec);
    const double q3[3] = {k * (B.P[0] - kh[0]), k * (B.P[1] - kh[1]), k * (B.P[2] - kh[2])};
    double F[2];
    tri_ff(B, dot3(q3, B.ex), dot3(q3, B.ey), F);
    const double k1 = dot3(kh, B.ex), k2 = dot3(kh, B.ey), k3 = dot3(kh, B.ez);
    const double k2c = fabs(k2) > K2CLAMP ? copysign(K2CLAMP, k2) : k2;
    const double sq = sqrt(1.0 - k2c * k2c), s13 = sqrt(1.0 - k2 * k2);
    double hv0 = kh[1], hv1 = -kh[0];
    if (!(fabs(kh[2]) < FWD_DOT)) {
        hv0 = yt - B.c[1];
        hv1 = -(xt - B.c[0]);
    }
    const double nh = sqrt(hv0 * hv0 + hv1 * hv1);
    const double hc[3] = {hv0 / nh, hv1 / nh, 0.0};
    double mvec[3], uu[3];
    for (int i = 0; i < 3; i++) mvec[i] = (B.ey[i] - k2c * kh[i]) / sq;
    cross3(kh, B.ey, uu);
    const double p = dot3(hc, mvec), qh = dot3(hc, uu) / s13;
    const double da = -0.5 * (B.Kz * sq + k3 / sq), db = -0.5 * k1 * k2c / sq;
    const double g = p * da + qh * db, h = p * db - qh * da;
    const double EFr = Ec * F[0] - Es * F[1], EFi = Ec * F[1] + Es * F[0];
    const double sr = -EFi / lambda, si = EFr / lambda;
    // (g I + h J) C: row 1 = g C1 + h C2, row 2 = g C2 - h C1
    for (int cc = 0; cc < 2; cc++) {
        const int i1 = 2 * (0 + 2 * cc), i2 = 2 * (1 + 2 * cc);
        const double r1r = g * B.C[i1] + h * B.C[i2], r1i = g * B.C[i1 + 1] + h * B.C[i2 + 1];
        const double r2r = g * B.C[i2] - h * B.C[i1], r2i = g * B.C[i2 + 1] - h * B.C[i1 + 1];
        acc[i1] += sr * r1r - si * r1i;
        acc[i1 + 1] += sr * r1i + si * r1r;
        acc[i2] += sr * r2r - si * r2i;
        acc[i2 + 1] += sr * r2i + si * r2r;
    }
}

// after the beam sum of model_bin_fp64: x T_phi, then e^{i k |x|}
__host__ __device__ inline void model_finish(double acc[8], double cp, double sp, double kr_rev)
{
    apply_temp_rot1(acc, cp, sp);
    apply_bin_phase(acc, kr_rev);
}

// Mixed-precision adjoint body: the geometry, q and every phase in FP64 (reduced to a
// half period before FP32 polynomials), the form factor's edge terms, the
// polarisation and its adjoint in FP32, the accumulators in FP64.  Near q -> 0 an
// FP32 series of the form factor and its gradient.  Edge phases come from the three vertex half-phase
// exponentials w_l = e^{i alpha_l / 2}: e^{i mu_j} = w_j w_{j+1},
// e^{i K_j / 2} = w_{j+1} conj(w_j); sinc(K_j / 2) from its series for |K_j| < 1.
// Mixed body: FP64 geometry, q and phases; the far-field phase e^{i k rho} is folded into
// the vertex exponentials, so F and dF/dq below carry it (F' = e^{i k rho} F); FP32
// elsewhere; contributions go to FP32 partial sums (the caller adds them into FP64 every
// ADJ_GROUP bins).  lam: Lam' of this bin in FP32.
__host__ __device__ inline void adj_bin_mixed(const AdjBeam& B, const AdjBin& bn, const float* __restrict__ lam,
                                              double waveno, double lambda, AdjAccF& acc)
{
    const double k = waveno;
    const double dx = bn.x - B.c[0], dy = bn.y - B.c[1], dz = bn.z - B.c[2];
    const double s2 = fma(dx, dx, fma(dy, dy, dz * dz));
    double y0 = (double)abt_rsqf((float)s2);
    double e = fma(-s2 * y0, y0, 1.0);
    y0 = fma(0.5 * y0, e, y0);
    e = fma(-s2 * y0, y0, 1.0);
    const double ir = fma(0.5 * y0, e, y0);              // 1 / rho
    const double kh[3] = {dx * ir, dy * ir, dz * ir};
    const double krev = k * 0.15915494309189535;
    const double kd = krev * (s2 * ir);                   // k rho / 2 pi
    const double q3[3] = {k * (B.P[0] - kh[0]), k * (B.P[1] - kh[1]), k * (B.P[2] - kh[2])};
    const double qx = fma(q3[0], B.ex[0], fma(q3[1], B.ex[1], q3[2] * B.ex[2]));
    const double qy = fma(q3[0], B.ey[0], fma(q3[1], B.ey[1], q3[2] * B.ey[2]));
    const float fqx = (float)qx, fqy = (float)qy;
    const float q2 = fmaf(fqx, fqx, fqy * fqy);
    float F[2], Gx[2], Gy[2];
    if ((double)q2 * B.qa2 < 2.25) {
        // FP32 series about q = 0 (|alpha_l| <= 1.5: 14 terms leave < 1e-9)
        float al[3];
        for (int l = 0; l < 3; l++) al[l] = fmaf(fqx, B.fxl[l], fqy * B.fyl[l]);
        const float e1 = al[0] + al[1] + al[2];
        const float e2 = fmaf(al[0], al[1], fmaf(al[1], al[2], al[2] * al[0]));
        const float e3 = al[0] * al[1] * al[2];
        float hm3 = 0.f, hm2 = 0.f, hm1 = 1.f, hprev = 1.f, inv = 0.5f;
        float d[3] = {0.f, 0.f, 0.f}, dr[3] = {0.f, 0.f, 0.f}, di[3] = {0.f, 0.f, 0.f};
        float fr = 0.5f, fi = 0.f;
        for (int n = 1; n <= 14; n++) {
            for (int l = 0; l < 3; l++) d[l] = fmaf(al[l], d[l], hprev);
            const float hn = fmaf(e1, hm1, fmaf(-e2, hm2, e3 * hm3));
            inv = inv / (float)(n + 2);
            const float t = hn * inv;
            switch (n & 3) {
                case 0: fr += t; for (int l = 0; l < 3; l++) dr[l] += d[l] * inv; break;
                case 1: fi += t; for (int l = 0; l < 3; l++) di[l] += d[l] * inv; break;
                case 2: fr -= t; for (int l = 0; l < 3; l++) dr[l] -= d[l] * inv; break;
                default: fi -= t; for (int l = 0; l < 3; l++) di[l] -= d[l] * inv; break;
            }
            hm3 = hm2; hm2 = hm1; hm1 = hn; hprev = hn;
        }
        const float A2 = (float)(2.0 * B.area);
        // times the far-field phase e^{i k rho}
        float Ec, Es;
        expi_pi(2.0 * kd, &Ec, &Es);
        const float Er = A2 * Ec, Ei = A2 * Es;
        const float gxr = dr[0] * B.fxl[0] + dr[1] * B.fxl[1] + dr[2] * B.fxl[2];
        const float gxi = di[0] * B.fxl[0] + di[1] * B.fxl[1] + di[2] * B.fxl[2];
        const float gyr = dr[0] * B.fyl[0] + dr[1] * B.fyl[1] + dr[2] * B.fyl[2];
        const float gyi = di[0] * B.fyl[0] + di[1] * B.fyl[1] + di[2] * B.fyl[2];
        F[0] = Er * fr - Ei * fi;
        F[1] = Er * fi + Ei * fr;
        Gx[0] = Er * gxr - Ei * gxi;
        Gx[1] = Er * gxi + Ei * gxr;
        Gy[0] = Er * gyr - Ei * gyi;
        Gy[1] = Er * gyi + Ei * gyr;
    } else {
        // vertex half phases alpha_l / 2 plus k rho / 2: w_l = e^{i pi t_l}, t_l = alpha_l / 2 pi + k rho / 2 pi
        float wr[3], wi[3];
        double al[3];
        for (int l = 0; l < 3; l++) {
            al[l] = fma(qx, B.xr[l], fma(qy, B.yr[l], kd));
            expi_pi(al[l], &wr[l], &wi[l]);
        }
        float sr = 0.f, si = 0.f, gxr = 0.f, gxi = 0.f, gyr = 0.f, gyi = 0.f;
        for (int j = 0; j < 3; j++) {
            const int jn = j == 2 ? 0 : j + 1;
            const float ex = B.fxl[jn] - B.fxl[j], ey = B.fyl[jn] - B.fyl[j];
            const float mx = 0.5f * (B.fxl[j] + B.fxl[jn]), my = 0.5f * (B.fyl[j] + B.fyl[jn]);
            const float x = 3.14159265358979f * (float)(al[jn] - al[j]);   // K_j / 2
            // e^{i x} = w_{j+1} conj(w_j), e^{i mu} = w_j w_{j+1}
            const float cx = wr[jn] * wr[j] + wi[jn] * wi[j];
            const float sx = wi[jn] * wr[j] - wr[jn] * wi[j];
            const float Er = wr[j] * wr[jn] - wi[j] * wi[jn];
            const float Ei = wr[j] * wi[jn] + wi[j] * wr[jn];
            const bool small = fabsf(x) < 0.5f;
            const float ix = abt_rcpf(x);
            const float Sq = sx * ix;
            const float S = small ? sinc_ser(x) : Sq;
            const float dS = 0.5f * (small ? dsinc_ser(x) : (cx - Sq) * ix);
            const float cj = B.fso * fmaf(fqx, ey, -fqy * ex);
            const float t = cj * S;
            sr = fmaf(t, Er, sr);
            si = fmaf(t, Ei, si);
            const float ax = fmaf(B.fso * ey, S, cj * dS * ex), ay = fmaf(-B.fso * ex, S, cj * dS * ey);
            gxr += ax * Er - t * mx * Ei;
            gxi += ax * Ei + t * mx * Er;
            gyr += ay * Er - t * my * Ei;
            gyi += ay * Ei + t * my * Er;
        }
        const float iq2 = abt_rcpf(q2);
        F[0] = -si * iq2;
        F[1] = sr * iq2;
        const float tx = 2.0f * fqx * iq2, ty = 2.0f * fqy * iq2;
        Gx[0] = -gxi * iq2 - tx * F[0];
        Gx[1] = gxr * iq2 - tx * F[1];
        Gy[0] = -gyi * iq2 - ty * F[0];
        Gy[1] = gyr * iq2 - ty * F[1];
    }
    // polarisation (FP32; the k_y clamp decided in FP64, as the reference does)
    const float kf[3] = {(float)kh[0], (float)kh[1], (float)kh[2]};
    const double k2d = fma(kh[0], B.ey[0], fma(kh[1], B.ey[1], kh[2] * B.ey[2]));
    const bool clamp = fabs(k2d) > K2CLAMP;
    const float k1 = fmaf(kf[0], B.fex[0], fmaf(kf[1], B.fex[1], kf[2] * B.fex[2]));
    const float k3 = fmaf(kf[0], B.fez[0], fmaf(kf[1], B.fez[1], kf[2] * B.fez[2]));
    const float k2 = (float)k2d;
    const float s13q = fmaf(k1, k1, k3 * k3);                    // 1 - k2^2
    const bool fb = !(fabs(kh[2]) < FWD_DOT);
    // Away from the clamp and the forward fallback, hc = unit(inc x khat) is normal to
    // khat, so hc.m = D' P0 and hc.unit(k x m) = D' Q0 with D' = rh / sqrt(1 - k2^2),
    // rh = 1 / |inc x khat|, P0 = e_y . (kh_y, -kh_x, 0), Q0 = e_y . ((inc.khat) khat - inc),
    // and g = D (P0 A + Q0 B), h = D (P0 B - Q0 A) with D = rh / (1 - k2^2),
    // A = -(K_z (1 - k2^2) + k3) / 2, B = -k1 k2 / 2.  P0, Q0 in FP64: both vanish at khat = +-e_y.
    const bool fast = !clamp && !fb;
    float g, h;
    float fP0 = 0.f, fQ0 = 0.f, fA = 0.f, fB = 0.f, fD = 0.f, rh = 0.f, is2 = 0.f;
    float k2c = 0.f, r13 = 0.f, s13 = 0.f, rsq = 0.f, sq = 0.f, inh = 0.f, hc0 = 0.f, hc1 = 0.f;
    float mv[3] = {0.f, 0.f, 0.f}, ev[3] = {0.f, 0.f, 0.f}, p = 0.f, qh = 0.f, da = 0.f, db = 0.f;
    if (fast) {
        fP0 = (float)fma(B.ey[0], kh[1], -B.ey[1] * kh[0]);
        fQ0 = (float)fma(-kh[2], k2d, B.ey[2]);
        rh = abt_rsqf(fmaf(kf[0], kf[0], kf[1] * kf[1]));
        is2 = abt_rcpf(s13q);
        fD = rh * is2;
        fA = -0.5f * fmaf(B.fKz, s13q, k3);
        fB = -0.5f * k1 * k2;
        g = fD * fmaf(fP0, fA, fQ0 * fB);
        h = fD * fmaf(fP0, fB, -fQ0 * fA);
    } else {
        k2c = clamp ? copysignf(0.99999898672103882f, k2) : k2;
        r13 = abt_rsqf(s13q);
        s13 = s13q * r13;
        const float sqq = clamp ? 2.02655679e-06f : s13q;
        rsq = clamp ? abt_rsqf(sqq) : r13;
        sq = sqq * rsq;
        float hvx, hvy;
        if (fb) {
            hvx = (float)(bn.yt - B.c[1]);
            hvy = (float)(-(bn.xt - B.c[0]));
        } else {
            hvx = kf[1];
            hvy = -kf[0];
        }
        inh = abt_rsqf(fmaf(hvx, hvx, hvy * hvy));
        hc0 = hvx * inh;
        hc1 = hvy * inh;
        const float uu[3] = {kf[1] * B.fey[2] - kf[2] * B.fey[1], kf[2] * B.fey[0] - kf[0] * B.fey[2],
                             kf[0] * B.fey[1] - kf[1] * B.fey[0]};
        for (int i = 0; i < 3; i++) {
            mv[i] = (B.fey[i] - k2c * kf[i]) * rsq;
            ev[i] = uu[i] * r13;
        }
        p = fmaf(hc0, mv[0], hc1 * mv[1]);
        qh = fmaf(hc0, ev[0], hc1 * ev[1]);
        da = -0.5f * fmaf(B.fKz, sq, k3 * rsq);
        db = -0.5f * k1 * k2c * rsq;
        g = fmaf(p, da, qh * db);
        h = fmaf(p, db, -qh * da);
    }
    // s = E (i / lambda) F  (F carries E)
    const float il = (float)(1.0 / lambda);
    const float sr = -F[1] * il, si = F[0] * il;
    float L[8];
    for (int q = 0; q < 8; q++) L[q] = lam[q];
    float z1r = 0.f, z1i = 0.f, z2r = 0.f, z2i = 0.f;
    for (int cc = 0; cc < 2; cc++) {
        const int i1 = 2 * (0 + 2 * cc), i2 = 2 * (1 + 2 * cc);
        const float l1r = L[i1], l1i = L[i1 + 1], l2r = L[i2], l2i = L[i2 + 1];
        const float c1r = B.fC[i1], c1i = B.fC[i1 + 1], c2r = B.fC[i2], c2i = B.fC[i2 + 1];
        z1r += l1r * c1r + l1i * c1i + l2r * c2r + l2i * c2i;
        z1i += l1r * c1i - l1i * c1r + l2r * c2i - l2i * c2r;
        z2r += l1r * c2r + l1i * c2i - (l2r * c1r + l2i * c1i);
        z2i += l1r * c2i - l1i * c2r - (l2r * c1i - l2i * c1r);
    }
    for (int cc = 0; cc < 2; cc++) {
        const int i1 = 2 * (0 + 2 * cc), i2 = 2 * (1 + 2 * cc);
        const float r1r = g * L[i1] - h * L[i2], r1i = g * L[i1 + 1] - h * L[i2 + 1];
        const float r2r = g * L[i2] + h * L[i1], r2i = g * L[i2 + 1] + h * L[i1 + 1];
        acc.GC[i1] += sr * r1r + si * r1i;
        acc.GC[i1 + 1] += sr * r1i - si * r1r;
        acc.GC[i2] += sr * r2r + si * r2i;
        acc.GC[i2 + 1] += sr * r2i - si * r2r;
    }
    const float gg = sr * z1r - si * z1i, gh = sr * z2r - si * z2i;
    const float mur = g * z1r + h * z2r, mui = g * z1i + h * z2i;
    // nu = mu E (i / lambda); E is in F and dF/dq
    const float nur = -mui * il, nui = mur * il;
    const float nFr = nur * F[0] - nui * F[1], nFi = nur * F[1] + nui * F[0];
    const float Rx = nur * Gx[0] - nui * Gx[1];
    const float Ry = nur * Gy[0] - nui * Gy[1];
    acc.S0 += nFr;
    for (int i = 0; i < 3; i++) {
        const float fq = (float)q3[i];
        acc.Qx[i] = fmaf(fq, Rx, acc.Qx[i]);
        acc.Qy[i] = fmaf(fq, Ry, acc.Qy[i]);
    }
    const float kw = (float)k;
    float kb[3];
    for (int i = 0; i < 3; i++) kb[i] = -kw * (Rx * B.fex[i] + Ry * B.fey[i]);
    float k1b, k2b, k3b, Kzb, eyb[3];
    float cbf[3] = {0.f, 0.f, 0.f};
    if (fast) {
        // reverse of g, h: the 1 - k2^2 inside A and D differentiated as a function of k2
        const float Pb = fD * fmaf(gg, fA, gh * fB);
        const float Qb = fD * fmaf(gg, fB, -gh * fA);
        const float Ab = fD * fmaf(gg, fP0, -gh * fQ0);
        const float Bb = fD * fmaf(gg, fQ0, gh * fP0);
        const float w = fmaf(gg, g, gh * h);                 // (dL/dD) D
        const float rw = w * rh * rh;
        Kzb = -0.5f * s13q * Ab;
        k3b = -0.5f * Ab;
        k1b = -0.5f * k2 * Bb;
        k2b = B.fKz * k2 * Ab - 0.5f * k1 * Bb + 2.f * k2 * w * is2 - kf[2] * Qb;
        kb[0] += -rw * kf[0] - B.fey[1] * Pb;
        kb[1] += -rw * kf[1] + B.fey[0] * Pb;
        kb[2] += -k2 * Qb;
        eyb[0] = kf[1] * Pb;
        eyb[1] = -kf[0] * Pb;
        eyb[2] = Qb;
    } else {
        const float pb = gg * da + gh * db, qb = gg * db - gh * da;
        const float dab = gg * p - gh * qh, dbb = gg * qh + gh * p;
        Kzb = -0.5f * sq * dab;
        float sqb = -0.5f * (B.fKz - k3 * rsq * rsq) * dab + 0.5f * k1 * k2c * rsq * rsq * dbb;
        k3b = -0.5f * dab * rsq;
        k1b = -0.5f * k2c * rsq * dbb;
        float k2cb = -0.5f * k1 * rsq * dbb;
        const float hcb0 = pb * mv[0] + qb * ev[0], hcb1 = pb * mv[1] + qb * ev[1];
        const float mb[3] = {pb * hc0, pb * hc1, 0.f};
        k2cb += -(mb[0] * kf[0] + mb[1] * kf[1]) * rsq;
        sqb += -(mb[0] * mv[0] + mb[1] * mv[1]) * rsq;
        const float ub[3] = {qb * hc0 * r13, qb * hc1 * r13, 0.f};
        const float s13b = -qb * (hc0 * ev[0] + hc1 * ev[1]) * r13;
        for (int i = 0; i < 3; i++) {
            eyb[i] = mb[i] * rsq;
            kb[i] += -k2c * rsq * mb[i];
        }
        // kb += e_y x ub; eyb += ub x khat  (ub has no z component)
        kb[0] += -B.fey[2] * ub[1];
        kb[1] += B.fey[2] * ub[0];
        kb[2] += B.fey[0] * ub[1] - B.fey[1] * ub[0];
        eyb[0] += ub[1] * kf[2];
        eyb[1] += -ub[0] * kf[2];
        eyb[2] += ub[0] * kf[1] - ub[1] * kf[0];
        k2b = -k2 * r13 * s13b;
        k2cb += -k2c * rsq * sqb;
        if (!clamp) k2b += k2cb;
        (void)s13;
        const float hdot = hcb0 * hc0 + hcb1 * hc1;
        const float hvbx = (hcb0 - hdot * hc0) * inh, hvby = (hcb1 - hdot * hc1) * inh;
        const float tx = -hvby, ty = hvbx;
        if (fb) {
            cbf[0] = -tx;
            cbf[1] = -ty;
        } else {
            kb[0] += tx;
            kb[1] += ty;
        }
    }
    for (int i = 0; i < 3; i++) {
        kb[i] += k1b * B.fex[i] + k2b * B.fey[i] + k3b * B.fez[i];
        acc.exb[i] += k1b * kf[i];
        acc.eyb[i] += eyb[i] + k2b * kf[i];
        acc.ezb[i] += k3b * kf[i] + Kzb * B.fP[i];
    }
    const float kk = kb[0] * kf[0] + kb[1] * kf[1] + kb[2] * kf[2];
    const float irf = (float)ir;
    const float ph = kw * nFi;
    for (int i = 0; i < 3; i++) acc.cb[i] += cbf[i] - (kb[i] - kk * kf[i]) * irf + ph * kf[i];
}

// Per-beam gradients from the accumulated sums: gv[9] = dL/dv_l (x,y,z per vertex, the
// record's vertex order), ga[8] = dL/d ampl (re/im pairs, the beam's own sign).
// u: the centre-relative vertices (record R_V20), P the propagation vector.
__host__ __device__ inline void adj_finish(const AdjBeam& B, const double* __restrict__ u, double sigma,
                                           const AdjAcc& acc, double* gv, double* ga)
{
    const double v0[3] = {u[0], u[1], u[2]}, v1[3] = {u[3], u[4], u[5]}, v2[3] = {u[6], u[7], u[8]};
    double a[3], b[3], N[3];
    for (int i = 0; i < 3; i++) { a[i] = v1[i] - v0[i]; b[i] = v2[i] - v0[i]; }
    cross3(a, b, N);
    const double nN = sqrt(dot3(N, N));
    const double n[3] = {N[0] / nN, N[1] / nN, N[2] / nN};
    // frame: e_x = e_y x e_z, e_y = w / |w|, w = e_z x P, e_z = -n
    double eyb[3], ezb[3], t[3];
    cross3(B.ez, acc.exb, t);
    for (int i = 0; i < 3; i++) eyb[i] = acc.eyb[i] + t[i];
    cross3(acc.exb, B.ey, t);
    for (int i = 0; i < 3; i++) ezb[i] = acc.ezb[i] + t[i];
    double w[3];
    cross3(B.ez, B.P, w);
    const double nw = sqrt(dot3(w, w));
    const double eye = dot3(eyb, B.ey);
    double wb[3];
    for (int i = 0; i < 3; i++) wb[i] = (eyb[i] - eye * B.ey[i]) / nw;
    cross3(B.P, wb, t);
    for (int i = 0; i < 3; i++) ezb[i] += t[i];
    const double ezn = dot3(ezb, n);
    double Nb[3];
    for (int i = 0; i < 3; i++) Nb[i] = -(ezb[i] - ezn * n[i]) / nN;
    // N = a x b
    double ab[3], bb[3];
    cross3(b, Nb, ab);
    cross3(Nb, a, bb);
    const double* V[3] = {v0, v1, v2};
    for (int l = 0; l < 3; l++) {
        const double* p1 = V[l == 2 ? 0 : l + 1];
        const double* p2 = V[l == 0 ? 2 : l - 1];
        double e[3], al[3];
        for (int i = 0; i < 3; i++) e[i] = p1[i] - p2[i];
        cross3(e, n, al);
        for (int i = 0; i < 3; i++) al[i] /= nN;
        const double ax = dot3(al, B.ex), ay = dot3(al, B.ey);
        for (int i = 0; i < 3; i++)
            gv[3 * l + i] = acc.S0 * al[i] + acc.Qx[i] * ax + acc.Qy[i] * ay + acc.cb[i] / 3.0;
    }
    for (int i = 0; i < 3; i++) {
        gv[3 + i] += ab[i];
        gv[6 + i] += bb[i];
        gv[i] -= ab[i] + bb[i];
    }
    for (int q = 0; q < 8; q++) ga[q] = sigma * acc.GC[q];
}

}  // namespace abt
