// ffbody.h -- per (beam, bin) bodies of the far-field kernels (far_field.hip).
// __host__ __device__ so that the same code also runs in the CPU emulator
// used by the tests (tests/emu); on the device abt_rsqf is the hardware
// reciprocal square root.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "records.h"
#include "trig.h"

namespace abt {

__host__ __device__ __forceinline__ float abt_rsqf(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsqf(x);
#else
    return 1.0f / sqrtf(x);
#endif
}

struct BinIn {
    double x, y, z;      // bin position
    double xt, yt, zt;   // bin (same phi, theta_i): forward fallback of the hc vector
    double rad;          // |bin position| (FP64 model body only)
};

__host__ __device__ __forceinline__ float abt_rcpf(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}

// ---------------------------------------------------------------------------
// Mixed-precision kernel body.

__host__ __device__ __forceinline__ float flipsign(float x, unsigned sgn)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __uint_as_float(__float_as_uint(x) ^ sgn);
#else
    unsigned u;
    memcpy(&u, &x, 4);
    u ^= sgn;
    memcpy(&x, &u, 4);
    return x;
#endif
}

// Polynomials in half revolutions: for |x| <= 1/2 and z = x^2,
//   sinpi_over(z) = sin(pi x) / x,  cospi_poly(z) = cos(pi x),  sincpi_poly(z) = sin(pi x) / (pi x);
// the coefficients of sin(2 pi r) / r and cos(2 pi r) (trig.h) scaled by powers of two.
__host__ __device__ __forceinline__ float sinpi_over(float z)
{
    return fmaf(z, fmaf(z, fmaf(z, fmaf(z, ABT_HR4 / 512.f, ABT_HR3 / 128.f), ABT_HR2 / 32.f), ABT_HR1 / 8.f),
                ABT_HR0 / 2.f);
}
__host__ __device__ __forceinline__ float cospi_poly(float z)
{
    return fmaf(z, fmaf(z, fmaf(z, fmaf(z, fmaf(z, ABT_KR5 / 1024.f, ABT_KR4 / 256.f), ABT_KR3 / 64.f),
                                ABT_KR2 / 16.f), ABT_KR1 / 4.f), ABT_KR0);
}
__host__ __device__ __forceinline__ float sincpi_poly(float z)
{
    constexpr double c = 0.15915494309189535;   // 1 / 2 pi
    return fmaf(z, fmaf(z, fmaf(z, fmaf(z, (float)(ABT_HR4 * c / 256.), (float)(ABT_HR3 * c / 64.)),
                                (float)(ABT_HR2 * c / 16.)), (float)(ABT_HR1 * c / 4.)), (float)(ABT_HR0 * c));
}

// t (FP64, half revolutions: e^{i pi t}) reduced to |x| <= 1/2: e^{i pi t} = (-1)^m e^{i pi x},
// m = rint(t); the parity of m comes back as an FP32 sign mask (bit 31).
__host__ __device__ __forceinline__ float pi_reduce(double t, unsigned* sgn)
{
    const double m = rint(t);
    *sgn = ((unsigned)(int)m) << 31;
    return (float)(t - m);
}

// e^{i pi t} in FP32 from the FP64 t
__host__ __device__ __forceinline__ void expi_pi(double t, float* c, float* s)
{
    unsigned sg;
    const float x = pi_reduce(t, &sg);
    const float z = x * x;
    *s = flipsign(x * sinpi_over(z), sg);
    *c = flipsign(cospi_poly(z), sg);
}

// An integer field of a beam record (the same in every lane of a wave) in a scalar register, so that
// branches on it are scalar and a polygon's vertex records come through scalar loads.
__host__ __device__ __forceinline__ int record_int(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_readfirstlane((int)x);
#else
    return (int)x;
#endif
}

// A whole number of a beam record, below 2^52, in scalar registers: the upper 32 bits, then the rest, both exact.  Read
// out of the bits of a sum with 2^52 instead, the polygons' branch took registers from the triangles': one orientation
// x 162,360 bins 4.97 ms, 4.63 so.
__host__ __device__ __forceinline__ int64_t record_int64(double x)
{
    uint32_t hi = (uint32_t)(x * 0x1p-32), lo = (uint32_t)fma(-0x1p32, (double)hi, x);
#if defined(__HIP_DEVICE_COMPILE__)
    hi = __builtin_amdgcn_readfirstlane(hi);
    lo = __builtin_amdgcn_readfirstlane(lo);
#endif
    return (int64_t)((uint64_t)hi << 32 | lo);
}

// x == 3.0 for a value that is the same in every lane of a wave, as a scalar condition
__host__ __device__ __forceinline__ bool record_is3(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_readfirstlane((int)(__builtin_bit_cast(uint64_t, x) >> 32)) == 0x40080000;
#else
    return x == 3.0;
#endif
}

// a <= b for two values that are the same in every lane of a wave, as a scalar condition
__host__ __device__ __forceinline__ bool record_less(double a, double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(a <= b) != 0;
#else
    return a <= b;
#endif
}

constexpr float SERIES_QA2 = 2.25f;  // (|q_perp| a)^2 below which the FP64 series is used
constexpr int SERIES_N = 16;         // truncation < 3e-12 relative at |q| a = 1.5

// 2 * sum_n i^n h_n(a,b,c) / (n+2)!  (triangle form factor / area, vertex phases a,b,c rad)
__host__ __device__ __forceinline__ void tri_series(double a, double b, double c, double* re, double* im)
{
    const double e1 = a + b + c;
    const double e2 = a * b + b * c + c * a;
    const double e3 = a * b * c;
    double h0 = 1.0, h1 = e1, h2 = e1 * e1 - e2;
    double inv = 0.5;             // 1/(n+2)! at n = 0
    double sr = h0 * inv, si = 0.0;
    inv = inv / 3.0;              // n = 1
    si += h1 * inv;
    inv = inv / 4.0;              // n = 2
    sr -= h2 * inv;
    double hm3 = h0, hm2 = h1, hm1 = h2;
#pragma unroll
    for (int n = 3; n <= SERIES_N; n++) {
        const double hn = e1 * hm1 - e2 * hm2 + e3 * hm3;
        inv = inv / (double)(n + 2);
        const double t = hn * inv;
        switch (n & 3) {
            case 0: sr += t; break;
            case 1: si += t; break;
            case 2: sr -= t; break;
            default: si -= t; break;
        }
        hm3 = hm2; hm2 = hm1; hm1 = hn;
    }
    *re = 2.0 * sr;
    *im = 2.0 * si;
}

// One edge of the rotation-invariant form factor with the far-field phase folded in:
// c_j sinc(pi d) e^{i (mu_j + k|r - com|)}, from the vertex exponentials w = e^{i pi t'}
// (t' = q.v + k|r - com|/2pi, half revolutions) of its two ends; d = t'_{j+1} - t'_j.
__host__ __device__ __forceinline__ void edge_exp(float wr0, float wi0, float wr1, float wi1, float d, float fqx,
                                                  float fqy, float edx, float edy, float& ssr, float& ssi)
{
    const float Er = fmaf(wr0, wr1, -wi0 * wi1);
    const float Ei = fmaf(wr0, wi1, wi0 * wr1);
    const float sx = fmaf(wi1, wr0, -wr1 * wi0);        // sin(pi d) = Im(w1 conj(w0))
    const float S = fabsf(d) < 0.5f ? sincpi_poly(d * d) : sx * abt_rcpf(3.14159265358979f * d);
    const float t = fmaf(fqx, edy, -fqy * edx) * S;
    ssr = fmaf(t, Er, ssr);
    ssi = fmaf(t, Ei, ssi);
}

// A record's FP32 blocks, in the address space of the record.
template <class Rec>
struct FloatsOf {
    typedef const float* type;
};
#if defined(__HIP_DEVICE_COMPILE__)
template <>
struct FloatsOf<const __attribute__((address_space(4))) double*> {
    typedef const __attribute__((address_space(4))) float* type;
};
#endif


// Mixed-precision body: one beam, one bin.  Adds the beam's contribution to the FP32
// projector sums accf: S+ (accf[0..3]) and S- (accf[4..7]), see mixed_finish; callers
// add accf into FP64 sums every few beams.  INC: also adds the squared Frobenius norm of
// the beam's amplitude, |f|^2 (gg^2 + hh^2) |A|_F^2 (the incoherent sum), to inc.
template <bool INC, class Rec>
__host__ __device__ __forceinline__ void beam_bin_mixed_t(Rec r, const double* __restrict__ vrecs,
                                                          const DevGrid& g, const BinIn& bi,
                                                          int fast_diff, float accf[8], float& inc)
{
    typedef typename FloatsOf<Rec>::type Floats;
    const Floats rf = (Floats)(r + R_F32), rg = (Floats)(r + R_G32);
    // ---- FP64 geometry: bin direction from the aperture centre, |r - com| ----
    const double dx = bi.x - r[R_COM], dy = bi.y - r[R_COM + 1], dz = bi.z - r[R_COM + 2];
    const double s = fma(dx, dx, fma(dy, dy, dz * dz));
    double y0 = (double)abt_rsqf((float)s);
    double e = fma(-s * y0, y0, 1.0);
    y0 = fma(0.5 * y0, e, y0);
    e = fma(-s * y0, y0, 1.0);
    const double invd = fma(0.5 * y0, e, y0);          // 1/|r - com|
    const double ux = dx * invd, uy = dy * invd, uz = dz * invd;
    if (fast_diff) {
        if (ux * r[R_PROP0] + uy * r[R_PROP0 + 1] + uz * r[R_PROP0 + 2] < r[R_COSFOV]) return;
    }
    // q = krev (prop2 - khat) in the aperture plane (revolutions per um); krev khat_x,y
    const Rec K = r + R_KRR;
    const double qx = fma(-K[0], ux, fma(-K[1], uy, fma(-K[2], uz, r[R_KP2])));
    const double qy = fma(-K[3], ux, fma(-K[4], uy, fma(-K[5], uz, r[R_KP2 + 1])));
    const double k1r = r[R_KP2] - qx, k2r = r[R_KP2 + 1] - qy;
    const double kd = g.krev * (s * invd);               // k |r - com| / 2 pi
    const float fqx = (float)qx, fqy = (float)qy;
    const float q2 = fmaf(fqx, fqx, fqy * fqy);
    const float il = g.inv_lambda_f;

    // ---- aperture integral with the far-field phase: (fR, fI) = e^{i k|r-com|} sum_ref / lambda ----
    float fR, fI;
    const bool tri = rf[F_NV] == 3.0f;
    if (q2 * rf[F_QA2] < SERIES_QA2) {
        // FP64 series of the form factor about q = 0; sum_ref = -i * (signed-area F)
        const double tw = 6.283185307179586;
        double sr = 0.0, si = 0.0;
        if (tri) {
            const double a = tw * fma(qx, r[R_EX], qy * r[R_EY]);
            const double b = tw * fma(qx, r[R_EX + 1], qy * r[R_EY + 1]);
            const double c = tw * fma(qx, r[R_EX + 2], qy * r[R_EY + 2]);
            double tr, ti;
            tri_series(a, b, c, &tr, &ti);
            sr = r[R_AREA] * tr;
            si = r[R_AREA] * ti;
        } else {
            const int nv = (int)rf[F_NV];
            const double* vr = vrecs + (int64_t)r[R_VOFF] * VREC;
            for (int j = 0; j < nv; j++) {
                const int jp = (j == nv - 1) ? 0 : j + 1;
                const double xj = vr[VREC * j + V_X], yj = vr[VREC * j + V_Y];
                const double xn = vr[VREC * jp + V_X], yn = vr[VREC * jp + V_Y];
                const double a = tw * fma(qx, xj, qy * yj);
                const double b = tw * fma(qx, xn, qy * yn);
                const double sa = 0.5 * (xj * yn - xn * yj);   // signed area of (com, j, j+1)
                double tr, ti;
                tri_series(0.0, a, b, &tr, &ti);
                sr += sa * tr;
                si += sa * ti;
            }
        }
        const float fr_ = (float)si, fi_ = (float)(-sr);
        float cb, sb;
        expi_pi(2.0 * kd, &cb, &sb);
        fR = (cb * fr_ - sb * fi_) * il;
        fI = (cb * fi_ + sb * fr_) * il;
    } else {
        // sum_ref = -(1/2pi) sum_j c_j sinc(pi d_j) e^{i mu_j} / |q|^2 (Fraunhofer, rotation-invariant form)
        float ssr = 0.f, ssi = 0.f;
        if (tri) {
            double t[3];
            float wr[3], wi[3];
#pragma unroll
            for (int l = 0; l < 3; l++) {
                t[l] = fma(qx, r[R_EX + l], fma(qy, r[R_EY + l], kd));
                expi_pi(t[l], &wr[l], &wi[l]);
            }
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const int jn = j == 2 ? 0 : j + 1;
                edge_exp(wr[j], wi[j], wr[jn], wi[jn], (float)(t[jn] - t[j]), fqx, fqy, rf[F_EDX + j],
                         rf[F_EDY + j], ssr, ssi);
            }
        } else {
            const int nv = (int)rf[F_NV];
            const double* vr = vrecs + (int64_t)r[R_VOFF] * VREC;
            const double t0 = fma(qx, vr[V_X], fma(qy, vr[V_Y], kd));
            float wr0, wi0;
            expi_pi(t0, &wr0, &wi0);
            double tp = t0;
            float wrp = wr0, wip = wi0;
            for (int j = 0; j < nv; j++) {
                double tn = t0;
                float wrn = wr0, win = wi0;
                if (j < nv - 1) {
                    tn = fma(qx, vr[VREC * (j + 1) + V_X], fma(qy, vr[VREC * (j + 1) + V_Y], kd));
                    expi_pi(tn, &wrn, &win);
                }
                edge_exp(wrp, wip, wrn, win, (float)(tn - tp), fqx, fqy, (float)vr[VREC * j + V_DX],
                         (float)vr[VREC * j + V_DY], ssr, ssi);
                tp = tn;
                wrp = wrn;
                wip = win;
            }
        }
        const float sc = (-0.15915494309189535f * il) * abt_rcpf(q2);
        fR = ssr * sc;
        fI = ssi * sc;
    }

    // ---- polarisation, FP32 (karczewski + rot4 of diff_mod.f90:124-198, 630-643) ----
    // rot4 . diff_ampl = gg I + hh J, J = [[0,1],[-1,0]]; the |k_y| > 0.999999 clamp
    // (diff_mod.f90:151) is decided in FP64, as the reference does
    const bool kclamp = fabs(k2r) > g.krev_k2clamp;
    const bool fwd = !(fabs(uz) < FWD_DOT);
    const float ik = g.inv_krev_f;
    const float fk1 = (float)k1r * ik, fk2 = (float)k2r * ik;
    // k_z in FP64: near k = +-e_y, 1 - k_y^2 = k_x^2 + k_z^2 is small and needs k_x, k_z to
    // relative (not absolute) FP32 precision
    const double* RR = r + R_RR;
    const float fk3 = (float)fma(RR[6], ux, fma(RR[7], uy, RR[8] * uz));
    const float s2 = fmaf(fk1, fk1, fk3 * fk3);                   // 1 - k_y^2 (unclamped)
    float gg, hh;
    if (!kclamp && !fwd) {
        // hc = unit(inc x khat) is normal to khat, so with m and k x m of karczewski:
        // hc.m = h_y / sqrt(1 - k_y^2), hc.unit(k x m) = (hc x khat)_y / sqrt(1 - k_y^2), where
        // |inc x khat| h_y = krow2 . (u_y, -u_x, 0) and |inc x khat| (hc x khat)_y = rr_23 - u_z k_y
        // (aperture frame, inc = (0,0,-1)); FP64 here, both vanish at k = +-e_y
        const double P0 = fma(K[3], uy, -K[4] * ux);       // krev |inc x khat| h_y
        const double Q0 = fma(-uz, k2r, K[5]);             // krev |inc x khat| (hc x khat)_y
        const float fux = (float)ux, fuy = (float)uy;
        const float rh = abt_rsqf(fmaf(fux, fux, fuy * fuy)) * abt_rcpf(s2);
        const float P = (float)P0 * rh, Q = (float)Q0 * rh;
        // diff_ampl(1,1) = (2,2) = A / sqrt(1 - k_y^2), diff_ampl(1,2) = -(2,1) = B / sqrt(1 - k_y^2)
        const float A = fmaf(rg[G_C1], s2, rg[G_C2] * fk3);
        const float B = fmaf(rg[G_C3], s2, rg[G_C2] * (fk1 * fk2));
        gg = fmaf(P, A, Q * B);
        hh = fmaf(P, B, -Q * A);
    } else {
        // clamped k_y, or the forward fallback of hc (diff_mod.f90:630-635): the bin
        // (same phi, theta_i); m and evo2 = unit(k x m) in closed form
        const float fk2c = kclamp ? copysignf(0.99999898672103882f, fk2) : fk2;
        const float s2c = kclamp ? 2.02655679e-06f : s2;        // clamped: 1 - 0.999999^2
        const float rs = abt_rsqf(s2c);
        const float sq = s2c * rs;                                 // sqrt(1 - k2^2)
        const float frac = sq * rf[F_SIG];
        const float ifrac = rs * rf[F_ISIG];
        float da = -0.5f * fmaf(rf[F_KZ], frac, fk3 * ifrac);          // diff_ampl(1,1) = (2,2)
        float db = 0.5f * fmaf(rf[F_KXY], frac, -fk1 * fk2c * ifrac);  // diff_ampl(1,2) = -(2,1)
        {
            // diff_ampl vanishes where k is the mirror image of prop2 in the aperture plane,
            // (k_x, k_y, k_z) = (K_x, K_y, -K_z): for every externally reflected beam that is
            // the forward direction, so thousands of beams share the zero there.  Through
            // dk = (k_x - K_x, k_y - K_y, k_z + K_z) (the first two from q, the third in FP64)
            // and u2 = k_y^2 - K_y^2 = dk_y (k_y + K_y), w2 = K_x dk_y + dk_x k_y:
            //   K_z (1 - k_y^2) + k_z (1 - K_y^2) = -K_z u2 + (1 - K_y^2) dk_z,
            //   K_x K_y (1 - k_y^2) - k_x k_y (1 - K_y^2) = -K_x K_y u2 - (1 - K_y^2) w2,
            // whose terms vanish with dk.  Used where |k_y| < 1/sqrt(2) (aperture frames put
            // prop2 in the x-z plane, K_y = 0, so that covers the zero); nearer k_y = +-1 the
            // terms of u2 outgrow 1 - k_y^2 and the direct form is kept.
            const float fdk1 = -fqx * ik, fdk2 = -fqy * ik;
            const float fdk3 = (float)fma(RR[6], ux, fma(RR[7], uy, fma(RR[8], uz, r[R_PROP2 + 2])));
            const float u2 = fdk2 * (fk2 + rf[F_KY]);
            const float w2 = fmaf(rf[F_KX], fdk2, fdk1 * fk2);
            const float dan = 0.5f * rs * fmaf(rf[F_KZ] * rf[F_SIG], u2, -rf[F_ISIG] * fdk3);
            const float dbn = -0.5f * rs * fmaf(rf[F_KXY] * rf[F_SIG], u2, rf[F_ISIG] * w2);
            const bool mir = !kclamp && s2 > 0.5f;
            da = mir ? dan : da;
            db = mir ? dbn : db;
        }
        const float m1 = -fk1 * fk2c * rs, m2 = sq, m3 = -fk2c * fk3 * rs;
        const float r13 = kclamp ? abt_rsqf(s2) : rs;
        const float ev1 = -fk3 * r13, ev3 = fk1 * r13;
        float hx = (float)uy, hy = (float)(-ux);
        if (fwd) {
            hx = (float)(bi.yt - r[R_COM + 1]);
            hy = (float)(-(bi.xt - r[R_COM]));
        }
        const float rh = abt_rsqf(fmaf(hx, hx, hy * hy));
        hx *= rh;
        hy *= rh;
        const float h1 = fmaf(rf[F_RR + 0], hx, rf[F_RR + 1] * hy);
        const float h2 = fmaf(rf[F_RR + 3], hx, rf[F_RR + 4] * hy);
        const float h3 = fmaf(rf[F_RR + 6], hx, rf[F_RR + 7] * hy);
        const float p = fmaf(h1, m1, fmaf(h2, m2, h3 * m3));
        const float qh = fmaf(h1, ev1, h3 * ev3);
        gg = fmaf(p, da, qh * db);
        hh = fmaf(p, db, -qh * da);
    }
    // f (gg I + hh J) = w P + w' Q with the projectors P, Q of J:  w = f (gg + i hh),
    // w' = f (gg - i hh);  P A = [r+; i r+],  Q A = [r-; -i r-]
    const float ta = fR * gg, tb = fI * hh, tc = fR * hh, td = fI * gg;
    const float wr = ta - tb, wi = tc + td, vr_ = ta + tb, vi = td - tc;
    if (INC) inc = fmaf(fmaf(fR, fR, fI * fI) * fmaf(gg, gg, hh * hh), rf[F_C2], inc);
    const float* rp = rg + G_RP;
    const float* rm = rg + G_RM;
    accf[0] = fmaf(wr, rp[0], fmaf(-wi, rp[1], accf[0]));
    accf[1] = fmaf(wr, rp[1], fmaf(wi, rp[0], accf[1]));
    accf[2] = fmaf(wr, rp[2], fmaf(-wi, rp[3], accf[2]));
    accf[3] = fmaf(wr, rp[3], fmaf(wi, rp[2], accf[3]));
    accf[4] = fmaf(vr_, rm[0], fmaf(-vi, rm[1], accf[4]));
    accf[5] = fmaf(vr_, rm[1], fmaf(vi, rm[0], accf[5]));
    accf[6] = fmaf(vr_, rm[2], fmaf(-vi, rm[3], accf[6]));
    accf[7] = fmaf(vr_, rm[3], fmaf(vi, rm[2], accf[7]));
}

__host__ __device__ __forceinline__ void beam_bin_mixed(const double* __restrict__ r,
                                                        const double* __restrict__ vrecs,
                                                        const DevGrid& g, const BinIn& bi,
                                                        int fast_diff, float accf[8])
{
    float unused = 0.f;
    beam_bin_mixed_t<false>(r, vrecs, g, bi, fast_diff, accf, unused);
}

// ---------------------------------------------------------------------------
// Restructured FP64 body: the mixed body's algorithm (bin direction from the aperture
// centre, rotation-invariant edge sum from vertex half-phase exponentials, the hc-normal
// polarisation closed form, projector accumulation) with every step in FP64.  Agrees with
// the reference's formula to ~1e-12 of the largest amplitude (the reference's own direct
// phase k |x3| ~ 1e7 rad carries ~1e-9 rad of rounding), at a fraction of its cost: three
// vertex exponentials per beam and bin instead of the split sum's twelve trigonometric
// pairs.  Used where the FP32 body's error would exceed the accuracy gate (the refinement
// pass of the mixed kernels) and as a fast FP64 precision of its own.

constexpr double PI64 = 3.141592653589793;

// Hardware approximations in FP64 (relative error below 2^-24 and 2^-24 on gfx950, measured on 10^9
// values); one costs as much as the FP32 one with its two conversions.
__host__ __device__ __forceinline__ double rcp_seed(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return 1.0 / x;
#endif
}
__host__ __device__ __forceinline__ double rsq_seed(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return 1.0 / sqrt(x);
#endif
}

// reciprocal and reciprocal square root to ~5e-15: one Newton step
__host__ __device__ __forceinline__ double rcp64_1(double x)
{
    const double y = rcp_seed(x);
    return fma(y, fma(-x, y, 1.0), y);
}
__host__ __device__ __forceinline__ double rsq64_1(double x)
{
    const double y = rsq_seed(x);
    return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}

// The functions below work on normal values whose squares and reciprocals are normal too, as the
// kernels' are, without the scaling that a general division or square root carries.

// 1 / x correctly rounded: two Newton steps from the approximation (2^-24 -> 2^-48 -> 2^-96 before
// the last rounding).  Equal to the IEEE quotient on 10^9 random values; 5 instructions for ~11.
__host__ __device__ __forceinline__ double rcp_cr(double x)
{
    double y = rcp_seed(x);
    y = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}

// 1 / x from an approximation y good to a few ulp, correctly rounded
__host__ __device__ __forceinline__ double rcp_from(double x, double y) { return fma(y, fma(-x, y, 1.0), y); }

// sqrt(s) from y = 1 / sqrt(s) to a few ulp, correctly rounded: the residual of s y decides the last bit
__host__ __device__ __forceinline__ double sqrt_from(double s, double y)
{
    const double g = s * y;
    return fma(fma(-g, g, s), 0.5 * y, g);
}

// sqrt(s) and the reciprocal of that root, both correctly rounded (10^9 random values): one coupled
// step for g = sqrt(s) and h = 1 / (2 g), then the residuals.
__host__ __device__ __forceinline__ double sqrt_cr(double s, double* inv)
{
    const double q = rsq_seed(s);
    double g = s * q, h = 0.5 * q;
    const double t = fma(-h, g, 0.5);
    g = fma(g, t, g);
    h = fma(h, t, h);
    g = fma(fma(-g, g, s), h, g);
    *inv = rcp_from(g, h + h);
    return g;
}

// 1 / sqrt(x) to ~1 ulp: one third-order step, e^3 ~ 2^-70
__host__ __device__ __forceinline__ double rsq64_3(double x)
{
    const double y = rsq_seed(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// The table of e^{i pi j / ETAB_N} (DevGrid::etab, ETAB_GRID doubles), built by the host in x87
// extended precision (64-bit significands): each angle reduced exactly to at most pi/4 (quarter
// turns, and the reflection a -> pi/2 - a within a quarter), so the extended-precision angle is
// within ~1e-19 of the exact one; cosine and sine rounded once to double, and the remainders (the
// low parts, at ETAB_LO).
inline void fill_exp_table(double* tab)
{
    const long double pi_l = 3.14159265358979323846264338327950288L;
    const int quarter = ETAB_N / 2;
    for (int j = 0; j < 2 * ETAB_N; j++) {
        const int q = j / quarter, m = j % quarter;
        const bool refl = 2 * m > quarter;
        const long double a = pi_l * (long double)(refl ? quarter - m : m) / (long double)ETAB_N;
        long double c = refl ? sinl(a) : cosl(a), s = refl ? cosl(a) : sinl(a);
        for (int k = 0; k < q; k++) {   // rotate by a quarter turn: (c, s) -> (-s, c)
            const long double t = c;
            c = -s;
            s = t;
        }
        const int i = 2 * j;
        tab[i] = (double)c;
        tab[i + 1] = (double)s;
        tab[ETAB_LO + i] = (double)(c - (long double)tab[i]);
        tab[ETAB_LO + i + 1] = (double)(s - (long double)tab[i + 1]);
    }
}

// What a caller of beam_bin_fp64r keeps after the table: the grid's far limit.
__host__ __device__ __forceinline__ void fp64r_constants(const DevGrid& g, double* c) { c[0] = g.cc_far; }

// e^{2 pi i T / (2 ETAB_N)} for an FP64 T in table steps (|T| < 2^31), from the table (in LDS on the device): T = J + r with
// J = rint(T) and |r| <= 1/2 (exact); the table holds the angle of J at index J mod 2 ETAB_N.  The rest
// is |y| <= pi / 1024: cos y from its Taylor polynomial (truncation below 2e-18), sin y from the cubic
// that is best in the largest error, y^5 / 120 replaced by its Chebyshev cubic (1.4e-16; a third
// coefficient would cost one instruction per exponential for less than the table's own rounding).
constexpr double EXP_H = 6.283185307179586 / (2.0 * ETAB_N);       // radians per step
constexpr double EXP_Y = 0.5 * EXP_H;                              // largest |y|
constexpr double EXP_S1 = EXP_H * (1.0 - EXP_Y * EXP_Y * EXP_Y * EXP_Y / 384.0);
constexpr double EXP_S3 = EXP_H * EXP_H * EXP_H * (-1.0 / 6.0 + EXP_Y * EXP_Y / 96.0);
constexpr double EXP_C2 = -0.5 * EXP_H * EXP_H;
constexpr double EXP_C4 = EXP_H * EXP_H * EXP_H * EXP_H / 24.0;
__host__ __device__ __forceinline__ void expi_step64(double T, const double* __restrict__ tab, double* c, double* s)
{
    const double jf = rint(T);
    const double r = T - jf;
    const int j = (int)jf & (2 * ETAB_N - 1);
    const double c0 = tab[2 * j], s0 = tab[2 * j + 1];
    const double w = r * r;
    const double sr = r * fma(w, EXP_S3, EXP_S1);
    const double cr = fma(w, fma(w, EXP_C4, EXP_C2), 1.0);
    *c = fma(c0, cr, -s0 * sr);
    *s = fma(s0, cr, c0 * sr);
}

// sin and cos of an FP64 angle x (radians, |x| < 2^40) from the same table with its low parts:
// x = n pi / ETAB_N + r with n = rint(x ETAB_N / pi), formed in the low bits of a 1.5 * 2^52
// shift, and r by a two-part Cody-Waite reduction (|r| <= pi / (2 ETAB_N) + 2^-30, error below
// 1e-18); e^{ix} = tab[n mod 2 ETAB_N] e^{ir}, the last from its Taylor polynomials (truncation
// below 2e-19 relative), the table entry taken as a double-double and the correction summed
// before its high part: ~0.5 ulp, the result rounded nearly correctly.  tab: ETAB_GRID doubles.
constexpr double SINCOS_SHIFT = 6755399441055744.0;                   // 1.5 * 2^52
constexpr double N_OVER_PI = (double)ETAB_N / 3.141592653589793;
constexpr double PI_OVER_N_HI = 3.141592653589793 / (double)ETAB_N;   // exact: a power-of-two scaling
constexpr double PI_OVER_N_LO = 1.2246467991473532e-16 / (double)ETAB_N;
struct SinCos {
    double c0, s0;   // the table's high parts
    double cl, sl;   // corrections: cos = c0 + cl, sin = s0 + sl
    __host__ __device__ __forceinline__ double c() const { return c0 + cl; }
    __host__ __device__ __forceinline__ double s() const { return s0 + sl; }
};
__host__ __device__ __forceinline__ SinCos sincos_parts64(double x, const double* __restrict__ tab)
{
    const double t = fma(x, N_OVER_PI, SINCOS_SHIFT);
    const double n = t - SINCOS_SHIFT;
    double r = fma(-n, PI_OVER_N_HI, x);
    r = fma(-n, PI_OVER_N_LO, r);
    const int j = (int)(uint32_t)__builtin_bit_cast(uint64_t, t) & (2 * ETAB_N - 1);
    SinCos o;
    o.c0 = tab[2 * j];
    o.s0 = tab[2 * j + 1];
    const double cl = tab[ETAB_LO + 2 * j], sl = tab[ETAB_LO + 2 * j + 1];
    const double z = r * r;
    const double sr = fma(r * z, fma(z, 1.0 / 120.0, -1.0 / 6.0), r);
    const double cm1 = z * fma(z, 1.0 / 24.0, -0.5);                   // cos r - 1
    o.sl = fma(o.c0, sr, fma(o.s0, cm1, sl));
    o.cl = fma(-o.s0, sr, fma(o.c0, cm1, cl));
    return o;
}
__host__ __device__ __forceinline__ void sincos_tab64(double x, const double* __restrict__ tab, double* s,
                                                      double* c)
{
    const SinCos v = sincos_parts64(x, tab);
    *s = v.s();
    *c = v.c();
}

// sin and cos of x + e, |e| <= SHIFT_MAX, from those of x: first order in e, summed into the
// corrections, so the result is rounded as sincos_tab64(x + e) is (e^2 / 2 < 5e-19).
constexpr double SHIFT_MAX = 9.313225746154785e-10;   // 2^-30
__host__ __device__ __forceinline__ void sincos_shift64(const SinCos& v, double c, double s, double e, double* se,
                                                        double* ce)
{
    *se = v.s0 + fma(e, c, v.sl);
    *ce = v.c0 + fma(-e, s, v.cl);
}

// a / b given y = 1 / b correctly rounded: q = a y, r = a - b q (exact), q + r y.  Equal to the
// IEEE quotient (Markstein's correction; no overflow or underflow in the kernels' ranges), at
// three operations per quotient once y is known.
__host__ __device__ __forceinline__ double div_by(double a, double b, double y)
{
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// f (gg I + hh J) A = w P A + w' Q A, w = f (gg + i hh), w' = f (gg - i hh)
template <class Rec>
__host__ __device__ __forceinline__ void add_projectors(Rec r, double FR, double FI, double gg, double hh, double acc[8])
{
    const double ta = FR * gg, tc = FR * hh;
    const double wr = fma(-FI, hh, ta), wi = fma(FI, gg, tc);
    const double vr = fma(FI, hh, ta), vi = fma(FI, gg, -tc);
    const Rec rp = r + R_RP64;
    const Rec rm = r + R_RM64;
    acc[0] = fma(wr, rp[0], fma(-wi, rp[1], acc[0]));
    acc[1] = fma(wr, rp[1], fma(wi, rp[0], acc[1]));
    acc[2] = fma(wr, rp[2], fma(-wi, rp[3], acc[2]));
    acc[3] = fma(wr, rp[3], fma(wi, rp[2], acc[3]));
    acc[4] = fma(vr, rm[0], fma(-vi, rm[1], acc[4]));
    acc[5] = fma(vr, rm[1], fma(vi, rm[0], acc[5]));
    acc[6] = fma(vr, rm[2], fma(-vi, rm[3], acc[6]));
    acc[7] = fma(vr, rm[3], fma(vi, rm[2], acc[7]));
}

// ---------------------------------------------------------------------------
// FP64 plain kernel body: one beam, one bin (diffraction, diff_mod.f90:576-670; karczewski
// :124-198; contour_integral :357-421).  Every input of a sine or cosine -- the bin offset
// and its rotation into the aperture frame, bvk = k |x3|, kxx and kyy with their clamps, and per
// edge delta, delta1, delta2, omega1, omega2 and the sums delta + omega -- is formed with the
// reference's operations in its order, without contraction, so the phases are the reference's
// doubles bit for bit: roots, reciprocals and quotients come from shorter sequences that equal the
// IEEE operations (sqrt_cr, rcp_cr, div_by).  Bound by FP64 VALU issue, so what is left out counts:
//   * the reference's ten sines and cosines per triangle need three table lookups besides bvk's:
//     delta_j + omega1 and delta_j + omega2 are both the phase of vertex j + 1 up to rounding
//     (~1e-14), so their values are delta_{j+1}'s moved by the exact difference (sincos_shift64),
//     rounded as their own lookups would be.  Clamped slopes (diff_mod.f90:379-382) move the phase
//     further: those edges look their own values up;
//   * the two roots |x1| and |x3| = |x1| (1 + rounding) share one hardware approximation, and the
//     reciprocals of both and of bvk follow from it.
// The amplitude algebra around the phases is reorganised; each step there changes a result by a
// few ulp at most:
//   * rot4 . diff_ampl = g I + h J (J = [[0,1],[-1,0]]: both factors have that form); away from the
//     k_y clamp and the forward fallback, hc = unit(inc x k) is normal to k, so with the Karczewski
//     vector m both come from one reciprocal root (the closed form of beam_bin_mixed);
//   * f (g I + h J) A summed through the projectors of J (beam_bin_mixed), which fp64_finish turns
//     into the amplitude matrix; temp_rot1 depends on phi only and is applied there too.
// The edge terms of contour_integral cancel one another, so they keep the reference's
// operations as well (the divisions included), in its order.
// The default column's diff_main (3702 beams x 64,980 bins): 630 VALU instructions and 6.5 ms of kernels
// before, 3.4 ms now; 5 orientations x 16,290 bins batched 7.9 -> 3.3 ms.
// acc: the projector sums S+ (0..3) and S- (4..7).  tab: the exponential table (LDS).
// INCOH: acc[0] += |amplC|_F^2 instead (temp_rot1 is orthogonal: the norm is final).
template <bool INCOH, class Rec>
__host__ __device__ __forceinline__ void beam_bin_fp64p(Rec r,
                                                        const double* __restrict__ vrecs,
                                                        const DevGrid& g, const BinIn& bi,
                                                        const double* __restrict__ tab, int fast_diff,
                                                        double acc[8])
{
#pragma clang fp contract(off)
    const double x1 = bi.x - r[R_COM], y1 = bi.y - r[R_COM + 1], z1 = bi.z - r[R_COM + 2];
    double ir1;
    const double r1 = sqrt_cr(x1 * x1 + y1 * y1 + z1 * z1, &ir1);
    if (fast_diff) {
        const double vx = div_by(x1, r1, ir1), vy = div_by(y1, r1, ir1), vz = div_by(z1, r1, ir1);
        if (vx * r[R_PROP0] + vy * r[R_PROP0 + 1] + vz * r[R_PROP0 + 2] < r[R_COSFOV]) return;
    }
    const Rec R = r + R_RR;
    const double x3 = R[0] * x1 + R[1] * y1 + R[2] * z1;
    const double y3 = R[3] * x1 + R[4] * y1 + R[5] * z1;
    const double z3 = R[6] * x1 + R[7] * y1 + R[8] * z1;
    const double Kx = r[R_PROP2], Ky = r[R_PROP2 + 1], Kz = r[R_PROP2 + 2];
    // the phase inputs of contour_integral (diff_mod.f90:357-375)
    const double w = g.waveno;
    const double bvk = w * sqrt_from(x3 * x3 + y3 * y3 + z3 * z3, ir1);
    const double ibvk = rcp_from(bvk, ir1 * g.inv_waveno);
    const double ww = w * w;
    double kxx = Kx * w - div_by(ww * x3, bvk, ibvk);
    double kyy = Ky * w - div_by(ww * y3, bvk, ibvk);
    if (fabs(kxx) < KMIN) kxx = KMIN;
    if (fabs(kyy) < KMIN) kyy = KMIN;
    // karczewski (diff_mod.f90:145-181): k = x3 / r1 as the reference divides, since k_y also
    // decides the clamp below
    const double k1 = div_by(x3, r1, ir1), k3 = div_by(z3, r1, ir1);
    const double k2 = div_by(y3, r1, ir1);
    const Rec C = r + R_C64;
    double gg, hj;   // rot4 . diff_ampl = gg I + hj J
    const double uz = z1 * ir1;
    // The reference's forward test is on inc . k with the clamped k_y (diff_mod.f90:151, 630).  Without the clamp
    // that is -uz to rounding, with it at most 1.02e-6 off: bins near the threshold (4.3e-6 and less below it, 9 in
    // the upper word) take the general branch, which forms it as the reference does.
    constexpr uint32_t near_fwd = (uint32_t)(__builtin_bit_cast(uint64_t, FWD_DOT) >> 32) - 9;
    const bool kclamp = fabs(k2) > K2CLAMP;
    const bool away = (uint32_t)(__builtin_bit_cast(uint64_t, fabs(uz)) >> 32) < near_fwd;
    if (!kclamp & away) {
        const double ux = x1 * ir1, uy = y1 * ir1;
        const double omk = fma(-k2, k2, 1.0);
        const double P0 = fma(R[3], uy, -(R[4] * ux));       // |inc x k| h_y
        const double Q0 = fma(-uz, k2, R[5]);                // |inc x k| (hc x k)_y
        const double rh = rsq64_3(fma(ux, ux, uy * uy) * (omk * omk));   // 1 / (|inc x k| (1 - k_y^2))
        const double P = P0 * rh, Q = Q0 * rh;
        const double A = fma(C[0], omk, C[1] * k3);
        const double B = fma(C[2], omk, C[1] * (k1 * k2));
        gg = fma(P, A, Q * B);
        hj = fma(P, B, -(Q * A));
    } else {
        const double k2c = kclamp ? copysign(K2CLAMP, k2) : k2;
        const double omk = fma(-k2c, k2c, 1.0);
        const double isq = rsq64_3(omk);                     // 1 / sqrt(1 - k2^2)
        const double k12 = k1 * k2c;
        const double m1 = -(k12 * isq), m2 = omk * isq, m3 = -(k2c * k3 * isq);
        const double frac = m2 * r[R_FRAC];                  // sqrt((1 - k2^2) / (1 - Ky^2))
        const double ifrac = isq * r[R_ISIG];                // its reciprocal
        const double a1m = -(Kz * frac), b2m = -(k3 * ifrac);
        const double b1m = fma(Kx * Ky, frac, -(k12 * ifrac));
        const double d11 = 0.5 * (a1m + b2m), d12 = 0.5 * b1m;   // diff_ampl = d11 I + d12 J
        // scattering-plane vector hc (diff_mod.f90:630-635) and rot4 = p I - qh J
        const double i1 = r[R_INC2], i2 = r[R_INC2 + 1], i3 = r[R_INC2 + 2];
        double kk1 = k1, kk2 = k2c, kk3 = k3;
        if (!(fabs(i1 * k1 + i2 * k2c + i3 * k3) < FWD_DOT)) {
            const double xt1 = bi.xt - r[R_COM], yt1 = bi.yt - r[R_COM + 1], zt1 = bi.zt - r[R_COM + 2];
            const double irt = rsq64_3(xt1 * xt1 + yt1 * yt1 + zt1 * zt1);
            kk1 = (R[0] * xt1 + R[1] * yt1 + R[2] * zt1) * irt;
            kk2 = (R[3] * xt1 + R[4] * yt1 + R[5] * zt1) * irt;
            kk3 = (R[6] * xt1 + R[7] * yt1 + R[8] * zt1) * irt;
        }
        const double h1 = fma(i2, kk3, -(i3 * kk2)), h2 = fma(i3, kk1, -(i1 * kk3)), h3 = fma(i1, kk2, -(i2 * kk1));
        const double e1 = fma(k2c, m3, -(k3 * m2)), e2 = fma(k3, m1, -(k1 * m3)), e3 = fma(k1, m2, -(k2c * m1));
        const double hh = fma(h1, h1, fma(h2, h2, h3 * h3));
        const double ee = fma(e1, e1, fma(e2, e2, e3 * e3));
        const double ihh = rsq64_3(hh);
        const double p = fma(h1, m1, fma(h2, m2, h3 * m3)) * ihh;
        const double qh = fma(h1, e1, fma(h2, e2, h3 * e3)) * (ihh * rsq64_3(ee));
        gg = fma(p, d11, qh * d12);
        hj = fma(p, d12, -(qh * d11));
    }
    // contour_integral (diff_mod.f90:357-421), edge by edge as the reference sums: the edge
    // terms cancel, so their roundings are kept too
    double sb, cb;
    sincos_tab64(bvk, tab, &sb, &cb);
    const double lam = g.lambda, ilam = g.inv_lambda;
    const double tkx = 2 * kxx, tky = 2 * kyy;
    double ar = 0.0, ai = 0.0;
    // one edge from vertex j (phase d0, sine and cosine s0, c0) to the next (phase dn, v its parts)
    const auto edge = [&](double d0, double s0, double c0, double dn, const SinCos& v, double sn, double cn,
                          double mj, double nj, double dx, double dy) {
#pragma clang fp contract(off)
        const double delta1 = kyy * mj + kxx;
        const double delta2 = kxx * nj + kyy;
        const double omega1 = dx * delta1;
        const double omega2 = dy * delta2;
        const double alpha = rcp_cr(tky * delta1);
        const double beta = rcp_cr(tkx * delta2);
        const double f1 = d0 + omega1, f2 = d0 + omega2;
        const double e1 = f1 - dn, e2 = f2 - dn;
        double s1, c1, s2, c2;
        sincos_shift64(v, cn, sn, e1, &s1, &c1);
        sincos_shift64(v, cn, sn, e2, &s2, &c2);
        if (!(fmax(fabs(e1), fabs(e2)) <= SHIFT_MAX)) {
            sincos_tab64(f1, tab, &s1, &c1);
            sincos_tab64(f2, tab, &s2, &c2);
        }
        const double sumim = alpha * (c0 - c1) - beta * (c0 - c2);
        const double sumre = -(alpha * (s0 - s1)) + beta * (s0 - s2);
        ar = ar + div_by(cb * sumre - sb * sumim, lam, ilam);
        ai = ai + div_by(cb * sumim + sb * sumre, lam, ilam);
    };
    // triangles: edges inline in the record; other vertex counts: a loop (polygons' vertex records)
    const int nv = record_int(r[R_NV]);
    if (nv == 3) {
        double d[3], s[3], c[3];
        SinCos v[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            d[j] = kxx * r[R_EX + j] + kyy * r[R_EY + j];
            v[j] = sincos_parts64(d[j], tab);
            s[j] = v[j].s();
            c[j] = v[j].c();
        }
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int n = j == 2 ? 0 : j + 1;
            edge(d[j], s[j], c[j], d[n], v[n], s[n], c[n], r[R_EM + j], r[R_EN + j], r[R_EDX + j], r[R_EDY + j]);
        }
    } else {
        const double* vr = vrecs + record_int64(r[R_VOFF]) * VREC;
        const auto field = [&](int j, int f, int inl) { return nv > 3 ? vr[VREC * j + f] : r[inl + j]; };
        const auto phase = [&](int j) {
#pragma clang fp contract(off)
            return kxx * field(j, V_X, R_EX) + kyy * field(j, V_Y, R_EY);
        };
        const double df = phase(0);
        const SinCos vf = sincos_parts64(df, tab);
        double d0 = df, s0 = vf.s(), c0 = vf.c();
        for (int j = 0; j < nv; j++) {
            const bool last = j == nv - 1;
            double dn = df;
            SinCos v = vf;
            if (!last) {
                dn = phase(j + 1);
                v = sincos_parts64(dn, tab);
            }
            const double sn = v.s(), cn = v.c();
            edge(d0, s0, c0, dn, v, sn, cn, field(j, V_M, R_EM), field(j, V_N, R_EN), field(j, V_DX, R_EDX),
                 field(j, V_DY, R_EDY));
            d0 = dn;
            s0 = sn;
            c0 = cn;
        }
    }
    if (INCOH) {
        // diagnostic: sum over beams of |amplC|_F^2 (conditioning of the coherent sum)
        double a2 = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) a2 = fma(r[R_AMPL + q], r[R_AMPL + q], a2);
        acc[0] = fma(a2 * fma(gg, gg, hj * hj), fma(ar, ar, ai * ai), acc[0]);
        return;
    }
    add_projectors(r, ar, ai, gg, hj, acc);
}

// From the projector sums to the amplitude matrix X = [S+ + S-; i (S+ - S-)], in place:
// re/im of (1,1) (2,1) (1,2) (2,2).
__host__ __device__ __forceinline__ void projectors_to_matrix(double a[8])
{
    const double x[8] = {a[0] + a[4], a[1] + a[5], -(a[1] - a[5]), a[0] - a[4],
                         a[2] + a[6], a[3] + a[7], -(a[3] - a[7]), a[2] - a[6]};
    for (int q = 0; q < 8; q++) a[q] = x[q];
}

// One beam, one bin of the plain body, added to the amplitude matrix acc (before temp_rot1): the CPU emulator's.
__host__ __device__ __forceinline__ void beam_bin_fp64(const double* __restrict__ r,
                                                       const double* __restrict__ vrecs,
                                                       const DevGrid& g, const BinIn& bi,
                                                       const double* __restrict__ tab, int fast_diff,
                                                       double acc[8])
{
    double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    beam_bin_fp64p<false>(r, vrecs, g, bi, tab, fast_diff, s);
    projectors_to_matrix(s);
    for (int q = 0; q < 8; q++) acc[q] += s[q];
}

// Difference form of one edge of the rotation-invariant form factor, from the full vertex
// phase exponentials W = e^{2 pi i t} of its two ends (t in revolutions):
//   c_j sinc(pi d) e^{i pi (t_j + t_{j+1})} = c_j (W_{j+1} - W_j) / (2 pi i d),  d = t_{j+1} - t_j,
// c_j = qx dy_j - qy dx_j.  Below |d| = 1e-3 (relative error of the difference there ~2e-16 /
// (pi |d|)) the product form with the Taylor polynomials of sinc(pi d) and e^{i pi d}, which
// only edges nearly normal to q reach.
__host__ __device__ __forceinline__ void edge_diff64(double Wr0, double Wi0, double Wr1, double Wi1, double d,
                                                     double qx, double qy, double edx, double edy, double& ssr,
                                                     double& ssi)
{
    const double c = fma(qx, edy, -qy * edx);
    if (fabs(d) >= 1e-3) {
        const double k = c * rcp64_1((2.0 * PI64) * d);
        ssr = fma(k, Wi1 - Wi0, ssr);       // c (W1 - W0) / (2 pi i d)
        ssi = fma(-k, Wr1 - Wr0, ssi);
    } else {
        const double x = PI64 * d, z = x * x;
        const double sinc = fma(z, fma(z, 1.0 / 120.0, -1.0 / 6.0), 1.0);
        const double ch = fma(z, fma(z, 1.0 / 24.0, -0.5), 1.0);          // e^{i pi d}
        const double sh = x * fma(z, fma(z, 1.0 / 120.0, -1.0 / 6.0), 1.0);
        const double k = c * sinc;
        ssr = fma(k, fma(Wr0, ch, -Wi0 * sh), ssr);
        ssi = fma(k, fma(Wr0, sh, Wi0 * ch), ssi);
    }
}

// What a lane keeps of its bin for the restructured FP64 body: the direction and 1 / distance.
struct FarBin {
    double nx, ny, nz, ir;
};
__host__ __device__ __forceinline__ FarBin far_bin(const BinIn& bi)
{
    const double ir = 1.0 / bi.rad;
    return {bi.x * ir, bi.y * ir, bi.z * ir, ir};
}

// Restructured FP64 body: one beam, one bin, added to the projector sums S+ (acc[0..3]) and
// S- (acc[4..7]) that fp64r_finish turns into the amplitude matrix.  Bound by FP64 VALU issue (one
// instruction of any kind takes 4 cycles of a SIMD); the common case -- a triangle seen away from its
// edges' nulls, its forward direction, the k_y clamp and the forward fallback -- is kept to 131 FP64
// instructions and 26 others (207 in all before):
//   * the far geometry: with h = (|c|^2 / 2 - x.c) / |x|^2 small, |x - c| - |x| and 1 / |x - c| are short
//     series in h -- no root, no reciprocal; their cut is checked per beam against the grid's limit
//     (g.cc_far, a scalar branch), beyond which both come from the distances;
//   * phases in table steps: the vertex coordinates carry krev and the table size, so a phase is
//     two FMAs and its table index is its rounding;
//   * one reciprocal root 1 / (|inc x k| (1 - k_y^2) |d0 d1 d2|) for the polarisation's normalisation
//     and the form factor's denominator together;
//   * records through scalar loads (k_sweep).
// Tried: the other branches after each tile in a pass of their own, which frees registers for a fifth wave but
// recomputes the beam (125 ms against 104; 112 with 4 waves).  Measured against the body before, each pair on one card
// (cards differ by up to 10 %), 24 orientations x 721 x 180 bins 112.7 -> 80.8 ms (1.8e10 beam.bins), 10,001 facets x
// 648,360 bins 40.5 -> 30.0 ms.
struct FarGeom {
    double ux, uy, uz;   // direction of the bin from the aperture centre
    double kd;           // k (|x - c| - |x|) in table steps (the bin's own e^{i k |x|} follows the beam sum)
    double id;           // 1 / |x - c|
};
// c: the centre, cc = |c|^2, kt: table steps per um; far: cc is within the far geometry's limit
template <class Rec>
__host__ __device__ __forceinline__ FarGeom far_geometry(Rec c, double cc, double kt, const FarBin& fb, bool far)
{
    FarGeom o;
    const double p = fma(fb.nx, c[0], fma(fb.ny, c[1], fb.nz * c[2]));
    if (far) {
        const double t = fma(0.5 * cc, fb.ir, -p);                   // |x| h
        const double h = t * fb.ir;
        // |x - c| = |x| sqrt(1 + 2 h): sqrt(1 + 2 h) - 1 = h (1 - h/2 + h^2/2 - 5/8 h^3 + ..),
        // 1 / sqrt(1 + 2 h) = 1 - h + 3/2 h^2 - 5/2 h^3 + ..
        o.kd = (kt * t) * fma(h, fma(h, fma(h, -0.625, 0.5), -0.5), 1.0);
        const double gd = fma(h, fma(h, fma(h, -2.5, 1.5), -1.0), 1.0);
        o.ux = fma(-c[0], fb.ir, fb.nx) * gd;
        o.uy = fma(-c[1], fb.ir, fb.ny) * gd;
        o.uz = fma(-c[2], fb.ir, fb.nz) * gd;
        o.id = fb.ir * gd;
    } else {
        // k (|x - c| - |x|) = k (|c|^2 - 2 x.c) / (|x - c| + |x|), formed without cancellation
        const double rad = rcp_cr(fb.ir);
        const double dx = fma(fb.nx, rad, -c[0]), dy = fma(fb.ny, rad, -c[1]), dz = fma(fb.nz, rad, -c[2]);
        const double s = fma(dx, dx, fma(dy, dy, dz * dz));
        o.id = rsq64_3(s);
        o.ux = dx * o.id;
        o.uy = dy * o.id;
        o.uz = dz * o.id;
        o.kd = kt * (fma(-2.0 * rad, p, cc) * rcp_cr(fma(s, o.id, rad)));
    }
    return o;
}

// Outside the beam's field of view (fast_diff; diff_mod.f90:593-603)
template <class Rec>
__host__ __device__ __forceinline__ bool far_culled(Rec r, const FarGeom& u, int fast_diff)
{
    return fast_diff && u.ux * r[R_PROP0] + u.uy * r[R_PROP0 + 1] + u.uz * r[R_PROP0 + 2] < r[R_COSFOV];
}

// The vertices' phases, exponentials and phase differences, in table steps.
struct TriPhase {
    double Wr[3], Wi[3], d0, d1, d2;
};
template <class Rec>
__host__ __device__ __forceinline__ TriPhase tri_phases_of(Rec tx, Rec ty, double q1, double q2, double kd,
                                                           const double* __restrict__ etab)
{
    TriPhase o;
    double T[3];
#pragma unroll
    for (int l = 0; l < 3; l++) {
        T[l] = fma(q1, tx[l], fma(q2, ty[l], kd));
        expi_step64(T[l], etab, &o.Wr[l], &o.Wi[l]);
    }
    o.d0 = T[1] - T[0];
    o.d1 = T[2] - T[1];
    o.d2 = T[0] - T[2];
    return o;
}
template <class Rec>
__host__ __device__ __forceinline__ TriPhase tri_phases(Rec r, double q1, double q2, double kd,
                                                        const double* __restrict__ etab)
{
    return tri_phases_of(r + R_TX, r + R_TY, q1, q2, kd, etab);
}

// One denominator: the form factor of a triangle is 2 A times the second divided difference of
// e^{i alpha} at its vertex phases alpha_l = 2 pi t_l, divided by i^2,
//   F = 2 A (W0 d1 + W1 d2 + W2 d0) / ((2 pi)^2 d0 d1 d2),  d_j = t_{j+1} - t_j,
// and sum_ref / lambda = -i F / lambda.  The exponentials' rounding enters the numerator as ~1.7e-16 max |d|, so
// F / A as ~9e-18 max |d| / |d0 d1 d2|: at most 1.7e-13 under the condition below (the two smaller |d_j| times
// each other at least 5e-5 turns^2: |d2| is at most twice the larger of the others), what the phases carry anyway (half an ulp of ~10^5 table steps is
// 5e-14 rad a vertex).  2 % of the waves have a lane beyond it (beams of the rough column); the earlier
// condition, every |d_j| >= 1e-3 and |q| a >= 1.5, left 13 % of them a lane in the other branch.
__host__ __device__ __forceinline__ bool one_denominator(const TriPhase& w, double d)
{
    // strict: q = 0 has every d_j = 0
    return fabs(d) > (1e-4 * (2 * ETAB_N) * (2 * ETAB_N)) * fmax(fabs(w.d0), fabs(w.d1));
}

// xt, yt: the theta_i bin of the same phi (forward fallback of hc).
template <class Rec>
__host__ __device__ __forceinline__ void beam_bin_fp64r_far(Rec r,
                                                            const double* __restrict__ vrecs, const FarBin& fb,
                                                            double xt, double yt, const double* __restrict__ etab,
                                                            double cc_far, int fast_diff, double acc[8])
{
    const FarGeom u = far_geometry(r + R_COM, r[R_CC], r[R_KT], fb, record_less(r[R_CC], cc_far));
    if (far_culled(r, u, fast_diff)) return;
    const Rec RR = r + R_RR;
    const double k1 = fma(RR[0], u.ux, fma(RR[1], u.uy, RR[2] * u.uz));
    const double k2 = fma(RR[3], u.ux, fma(RR[4], u.uy, RR[5] * u.uz));
    const double k3 = fma(RR[6], u.ux, fma(RR[7], u.uy, RR[8] * u.uz));
    const double q1 = r[R_PROP2] - k1, q2 = r[R_PROP2 + 1] - k2;   // q / k in the aperture plane
    const bool nv3 = record_is3(r[R_NV]);
    TriPhase w;
    double d = 0.0;
    bool one = false;
    if (nv3) {
        w = tri_phases(r, q1, q2, u.kd, etab);
        d = w.d0 * w.d1 * w.d2;
        one = one_denominator(w, d);
    }
    const bool kclamp = fabs(k2) > K2CLAMP, fwd = !(fabs(u.uz) < FWD_DOT);
    const double s2 = fma(k1, k1, k3 * k3);                        // 1 - k_y^2 (unclamped)
    // (FR, FI) = e^{i k (|x-c| - |x|)} sum_ref / lambda; gg I + hh J: karczewski + rot4 (diff_mod.f90:124-198,
    // 630-643)
    double FR, FI, gg, hh;
    if (one && !kclamp && !fwd) {
        // hc = unit(inc x khat) is normal to khat (see beam_bin_mixed)
        const Rec C = r + R_C64;
        const double P0 = fma(RR[3], u.uy, -RR[4] * u.ux);
        const double Q0 = fma(-u.uz, k2, RR[5]);
        const double m = s2 * d;
        const double ri = rsq64_1(fma(u.ux, u.ux, u.uy * u.uy) * (m * m));   // 1 / (|(ux, uy)| s2 |d|)
        const double f = r[R_TA] * copysign(ri, d);
        const double A = fma(C[0], s2, C[1] * k3);
        const double B = fma(C[2], s2, C[1] * (k1 * k2));
        FR = f * fma(w.Wi[0], w.d1, fma(w.Wi[1], w.d2, w.Wi[2] * w.d0));
        FI = -f * fma(w.Wr[0], w.d1, fma(w.Wr[1], w.d2, w.Wr[2] * w.d0));
        gg = fma(P0, A, Q0 * B);
        hh = fma(P0, B, -Q0 * A);
    } else {
        const double qx = r[R_KREV] * q1, qy = r[R_KREV] * q2;   // revolutions per um
        if (one) {
            const double f = r[R_TA] * rcp64_1(d);
            FR = f * fma(w.Wi[0], w.d1, fma(w.Wi[1], w.d2, w.Wi[2] * w.d0));
            FI = -f * fma(w.Wr[0], w.d1, fma(w.Wr[1], w.d2, w.Wr[2] * w.d0));
        } else if (fma(q1, q1, q2 * q2) * r[R_SA2] < (double)SERIES_QA2) {   // (|q| a)^2
            const double tw = 6.283185307179586;
            double sr = 0.0, si = 0.0;
            if (nv3) {
                const double a = tw * fma(qx, r[R_EX], qy * r[R_EY]);
                const double b = tw * fma(qx, r[R_EX + 1], qy * r[R_EY + 1]);
                const double c = tw * fma(qx, r[R_EX + 2], qy * r[R_EY + 2]);
                double tr, ti;
                tri_series(a, b, c, &tr, &ti);
                sr = r[R_AREA] * tr;
                si = r[R_AREA] * ti;
            } else {
                const int nv = record_int(r[R_NV]);
                const double* vr = vrecs + record_int64(r[R_VOFF]) * VREC;
                for (int j = 0; j < nv; j++) {
                    const int jp = (j == nv - 1) ? 0 : j + 1;
                    const double xj = vr[VREC * j + V_X], yj = vr[VREC * j + V_Y];
                    const double xn = vr[VREC * jp + V_X], yn = vr[VREC * jp + V_Y];
                    const double a = tw * fma(qx, xj, qy * yj);
                    const double b = tw * fma(qx, xn, qy * yn);
                    const double sa = 0.5 * (xj * yn - xn * yj);
                    double tr, ti;
                    tri_series(0.0, a, b, &tr, &ti);
                    sr += sa * tr;
                    si += sa * ti;
                }
            }
            // sum_ref = -i F = si - i sr
            double cb, sb;
            expi_step64(u.kd, etab, &cb, &sb);
            FR = (cb * si + sb * sr) * r[R_IL];
            FI = (sb * si - cb * sr) * r[R_IL];
        } else {
            constexpr double turn = 1.0 / (2 * ETAB_N);
            double ssr = 0.0, ssi = 0.0;
            if (nv3) {
                edge_diff64(w.Wr[0], w.Wi[0], w.Wr[1], w.Wi[1], turn * w.d0, qx, qy, r[R_EDX], r[R_EDY], ssr, ssi);
                edge_diff64(w.Wr[1], w.Wi[1], w.Wr[2], w.Wi[2], turn * w.d1, qx, qy, r[R_EDX + 1], r[R_EDY + 1], ssr, ssi);
                edge_diff64(w.Wr[2], w.Wi[2], w.Wr[0], w.Wi[0], turn * w.d2, qx, qy, r[R_EDX + 2], r[R_EDY + 2], ssr, ssi);
            } else {
                const int nv = record_int(r[R_NV]);
                const double* vr = vrecs + record_int64(r[R_VOFF]) * VREC;
                const double sx = (2 * ETAB_N) * qx, sy = (2 * ETAB_N) * qy;
                const double T0 = fma(sx, vr[V_X], fma(sy, vr[V_Y], u.kd));
                double Wr0, Wi0;
                expi_step64(T0, etab, &Wr0, &Wi0);
                double Tp = T0, Wrp = Wr0, Wip = Wi0;
                for (int j = 0; j < nv; j++) {
                    double Tn = T0, Wrn = Wr0, Win = Wi0;
                    if (j < nv - 1) {
                        Tn = fma(sx, vr[VREC * (j + 1) + V_X], fma(sy, vr[VREC * (j + 1) + V_Y], u.kd));
                        expi_step64(Tn, etab, &Wrn, &Win);
                    }
                    edge_diff64(Wrp, Wip, Wrn, Win, turn * (Tn - Tp), qx, qy, vr[VREC * j + V_DX], vr[VREC * j + V_DY],
                                ssr, ssi);
                    Tp = Tn;
                    Wrp = Wrn;
                    Wip = Win;
                }
            }
            const double sc = -r[R_IL] * rcp64_1(6.283185307179586 * fma(qx, qx, qy * qy));
            FR = ssr * sc;
            FI = ssi * sc;
        }
        if (!kclamp && !fwd) {
            const Rec C = r + R_C64;
            const double P0 = fma(RR[3], u.uy, -RR[4] * u.ux);
            const double Q0 = fma(-u.uz, k2, RR[5]);
            const double rh = rsq64_1(fma(u.ux, u.ux, u.uy * u.uy) * (s2 * s2));   // 1 / (|(ux, uy)| s2)
            const double P = P0 * rh, Q = Q0 * rh;
            const double A = fma(C[0], s2, C[1] * k3);
            const double B = fma(C[2], s2, C[1] * (k1 * k2));
            gg = fma(P, A, Q * B);
            hh = fma(P, B, -Q * A);
        } else {
            const double Kx = r[R_PROP2], Ky = r[R_PROP2 + 1], Kz = r[R_PROP2 + 2];
            const double sig = r[R_FRAC], isig = r[R_ISIG];
            const double k2c = kclamp ? copysign(K2CLAMP, k2) : k2;
            const double s2c = kclamp ? (1.0 - K2CLAMP * K2CLAMP) : s2;
            const double rs = rsq64_3(s2c);
            const double sq = s2c * rs;
            const double frac = sq * sig;
            const double ifrac = rs * isig;
            double da = -0.5 * fma(Kz, frac, k3 * ifrac);
            double db = 0.5 * fma(Kx * Ky, frac, -k1 * k2c * ifrac);
            {
                // the mirror-zero form (see beam_bin_mixed)
                const double dk3 = fma(RR[6], u.ux, fma(RR[7], u.uy, fma(RR[8], u.uz, Kz)));
                const double u2 = -q2 * (k2 + Ky);
                const double w2 = fma(Kx, -q2, -q1 * k2);
                const double dan = 0.5 * rs * fma(Kz * sig, u2, -isig * dk3);
                const double dbn = -0.5 * rs * fma(Kx * Ky * sig, u2, isig * w2);
                const bool mir = !kclamp && s2 > 0.5;
                da = mir ? dan : da;
                db = mir ? dbn : db;
            }
            const double m1 = -k1 * k2c * rs, m2 = sq, m3 = -k2c * k3 * rs;
            const double r13 = kclamp ? rsq64_3(s2) : rs;
            const double ev1 = -k3 * r13, ev3 = k1 * r13;
            double hx = u.uy, hy = -u.ux;
            if (fwd) {
                hx = yt - r[R_COM + 1];
                hy = -(xt - r[R_COM]);
            }
            const double rh = rsq64_3(fma(hx, hx, hy * hy));
            hx *= rh;
            hy *= rh;
            const double h1 = fma(RR[0], hx, RR[1] * hy);
            const double h2 = fma(RR[3], hx, RR[4] * hy);
            const double h3 = fma(RR[6], hx, RR[7] * hy);
            const double pm = fma(h1, m1, fma(h2, m2, h3 * m3));
            const double qh = fma(h1, ev1, h3 * ev3);
            gg = fma(pm, da, qh * db);
            hh = fma(pm, db, -qh * da);
        }
    }
    add_projectors(r, FR, FI, gg, hh, acc);
}

// One beam, one bin from the bin's plain inputs (bi.rad = |x| is read), for the CPU emulator of the bodies; etab: the
// table, then fp64r_constants.
__host__ __device__ __forceinline__ void beam_bin_fp64r(const double* __restrict__ r,
                                                        const double* __restrict__ vrecs,
                                                        const DevGrid& g, const BinIn& bi,
                                                        const double* __restrict__ etab,
                                                        int fast_diff, double acc[8])
{
    (void)g;
    beam_bin_fp64r_far(r, vrecs, far_bin(bi), bi.xt, bi.yt, etab, etab[ETAB_CC_FAR], fast_diff, acc);
}

// Beams per FP32 partial sum of the mixed kernels: every MIXED_GROUP consecutive beams
// (counted from the start of the beam list, or of the orientation) are summed in FP32 and
// the partial is added to the FP64 sums.  Tile sizes and chunk lengths are multiples of it,
// so the groups, and the result, do not depend on them.
constexpr int MIXED_GROUP = 8;

// The per-bin phase factor e^{i k |x|} of the FP64 model body (adjbody.h).
__host__ __device__ __forceinline__ void apply_bin_phase(double acc[8], double kr_rev)
{
#pragma clang fp contract(off)
    double s, c;
    sincos_f64(6.283185307179586 * (kr_rev - rint(kr_rev)), &s, &c);
    for (int q = 0; q < 4; q++) {
        const double re = acc[2 * q], im = acc[2 * q + 1];
        acc[2 * q] = re * c - im * s;
        acc[2 * q + 1] = re * s + im * c;
    }
}

// From the projector sums S+ = acc[0..3], S- = acc[4..7] (columns 1, 2) to the
// amplitude matrix, then temp_rot1 on the right.
__host__ __device__ __forceinline__ void apply_temp_rot1(double acc[8], double cp, double sp);

__host__ __device__ __forceinline__ void mixed_finish(double acc[8], double cp, double sp)
{
    projectors_to_matrix(acc);
    apply_temp_rot1(acc, cp, sp);
}

// The mixed kernel sums f_b G_b A_b over beams per bin; the phi-only rotation
// temp_rot1 = [[-s,-c],[c,-s]] (diff_mod.f90:646-650) is applied once on the right:
// (X T)(r,1) = -s X(r,1) + c X(r,2);  (X T)(r,2) = -c X(r,1) - s X(r,2).
__host__ __device__ __forceinline__ void apply_temp_rot1(double acc[8], double cp, double sp)
{
    double o[8];
    for (int rr = 0; rr < 2; rr++)
        for (int ri = 0; ri < 2; ri++) {
            const double x1 = acc[2 * rr + ri];        // X(r,1)
            const double x2 = acc[4 + 2 * rr + ri];    // X(r,2)
            o[2 * rr + ri] = fma(-sp, x1, cp * x2);
            o[4 + 2 * rr + ri] = fma(-cp, x1, -sp * x2);
        }
    for (int q = 0; q < 8; q++) acc[q] = o[q];
}

// After the beam sum of beam_bin_fp64r: the projector sums to the amplitude matrix (with
// temp_rot1), then the bin's far-field phase e^{i k |x|} (kr_rev = k |x| / 2 pi).
__host__ __device__ __forceinline__ void fp64r_finish(double acc[8], double cp, double sp, double kr_rev)
{
    mixed_finish(acc, cp, sp);
    apply_bin_phase(acc, kr_rev);
}

}  // namespace abt
