// kr_exact64.h -- the FP64 flux functions of the GPU kernels: the
// values of the reference's PLM and of the general hlld and hllc of
// kr_physics.h bit for bit, the sign of a zero aside, in fewer instructions
// and without branches.
//
// What bounds them is the number of FP64 instructions a wave issues; half of
// hlld<double> is IEEE divisions (31 of about 16 issue slots each, counting
// v_rcp_f64 as four).  A division is
//     scale n, d;  r = refined reciprocal of d;  q = n r;
//     q' = q + r (n - d q);  unscale, fix up zero / inf / nan
// and everything up to r depends on the denominator alone, so quotients over
// one denominator share it (hlld has 12 denominators), and 1 / (gamma - 1)
// and its inverse come from the host.  Leaving out the scaling changes no
// bit of a quotient while n is 0 or within 2^-968 .. 2^500 (below, the
// remainder n - d q needs bits under 2^-1074), d within 2^-240 .. 2^240 and
// the quotient is normal.  Inputs take the general function, a branch of the
// whole wave, when a velocity or field is below 2^-840 but not 0, an input is
// above 2^60 or not a number, or rho or p is below 2^-60.  Past that guard:
//   - numerators linear in a transverse velocity or in the field keep the
//     range.  The smallest are b_x (u* - u) in a star state and rho* v* in a
//     double star; u* - u, or the rotation that makes v* from a v = 0, is at
//     least 2^-53 of a wave speed above 2^-61, and rho* above 2^-62;
//   - numerators of second order (b_x^2, b_t^2, rho* v.b, b_x rho* u* + m.b)
//     may leave it, or vanish.  Their quotients are right to far better than
//     2^-900, and each ends in a sum with one that is exact and at least
//     2^-180: c_s^2 in both arguments of the speed's square roots, (s - u) e
//     and e* in the energies.  What is off lies below half an ulp of the sum.
//
// The branches of hlld<double> (flat slopes, degenerate star states, the
// region of the Riemann fan) become selects: with two waves on a SIMD the
// divisions' dependent chains are hidden only if independent ones are issued
// between them, which a branch around each prevents, and lanes of one wave
// take different branches anyway.  Past the star states only the side of the
// contact that the flux takes is evaluated.
#pragma once

#include "kr_physics.h"

namespace kr {

// n / d as the compiler expands it, written out so that it is not moved
// into a branch.
__device__ __forceinline__ double div64(double n, double d) {
    bool vcc, unused;
    const double ds = __builtin_amdgcn_div_scale(n, d, false, &unused);
    const double ns = __builtin_amdgcn_div_scale(n, d, true, &vcc);
    double r = __builtin_amdgcn_rcp(ds);
    r = __builtin_fma(r, __builtin_fma(-ds, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-ds, r, 1.0), r);
    const double q = ns * r;
    return __builtin_amdgcn_div_fixup(
        __builtin_amdgcn_div_fmas(__builtin_fma(-ds, q, ns), r, q, vcc), d, n);
}

// A denominator and its refined reciprocal; n / d for the range above.
struct Den64 {
    double d, r;
};
__device__ __forceinline__ Den64 den64(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
    return {d, r};
}
__device__ __forceinline__ double over64(double n, const Den64 &c) {
    const double q = n * c.r;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-c.d, q, n), c.r, q), c.d, n);
}

// PLM increments t of N cells or variables from their differences to the
// lower and upper neighbour, in the reference's expression order
// (hydro/reconstruct/plm.h:116-153; 0 where the differences disagree in
// sign): a cell's two face states are q + t and q - t.  All N divisions are
// issued side by side; a wave in which every slope is flat (a medium at rest
// around a blast) skips them.
template <int N>
__device__ __forceinline__ void plm_inc64(const double *lo, const double *hi, double *t) {
    double d[N];
    bool steep = false;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        d[k] = lo[k] * hi[k];
        steep |= !(d[k] <= 0);
        t[k] = 0;
    }
    if (!__any(steep)) return;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double coef = div64(d[k], lo[k] * lo[k] + hi[k] * hi[k] + d[k] * 2);
        const double inc = coef * (lo[k] + hi[k]);
        t[k] = d[k] <= 0 ? 0.0 : inc;
    }
}

// |x| as an ordered integer, its high word, with 0 the largest: the value
// is at least kSmall64 <=> x = 0 or |x| > 2^-840.  The shift takes in the low
// word: a subnormal below 2^-1042 has no other bits.
constexpr unsigned kSmall64 = (1023u - 840u) << 21;
__device__ __forceinline__ unsigned mag64(double x) {
    return (unsigned)((((unsigned long long)__double_as_longlong(x) << 1) - 1u) >> 32);
}
__device__ __forceinline__ unsigned umin3(unsigned a, unsigned b, unsigned c) {
    const unsigned d = a < b ? a : b;
    return d < c ? d : c;
}

struct Gam64 {
    double g;          // gamma
    double cv;         // 1 / (gamma - 1)
    double ge;         // 1 / cv + 1: the gamma that hlld's wave speeds use
};

template <class T> __device__ __forceinline__ T sel(bool c, T a, T b) { return c ? a : b; }

// hlld<double> (mhd/riemann/hlld.h:81-298) without the normal slot BCC:
// about 650 VALU instructions where the general function issues 1,000.
__device__ __forceinline__ void hlld64(double *flx, const double *wl, const double *wr, const Gam64 &k) {
    {
        // the sum is not a number if one of them is
        const double big = kfabs(wl[MOM]) + kfabs(wl[MOM + 1]) + kfabs(wl[MOM + 2]) + kfabs(wr[MOM]) +
                           kfabs(wr[MOM + 1]) + kfabs(wr[MOM + 2]) + kfabs(wl[BCC]) + kfabs(wl[BCC + 1]) +
                           kfabs(wl[BCC + 2]) + kfabs(wr[BCC + 1]) + kfabs(wr[BCC + 2]) + wl[RHO] +
                           wr[RHO] + wl[ENE] + wr[ENE];
        unsigned s = umin3(mag64(wl[MOM]), mag64(wr[MOM]), mag64(wl[BCC]));
        s = umin3(s, mag64(wl[MOM + 1]), mag64(wr[MOM + 1]));
        s = umin3(s, mag64(wl[MOM + 2]), mag64(wr[MOM + 2]));
        s = umin3(s, mag64(wl[BCC + 1]), mag64(wr[BCC + 1]));
        s = umin3(s, mag64(wl[BCC + 2]), mag64(wr[BCC + 2]));
        const double lo = 0x1p-60;
        const bool in = big < 0x1p60 && s >= kSmall64 && wl[RHO] > lo && wr[RHO] > lo && wl[ENE] > lo &&
                        wr[ENE] > lo;
        if (__builtin_expect(!__all(in), 0)) {
            hlld<double>(flx, wl, wr, k.g);
            return;
        }
    }
    const double bx = wl[BCC], bx2 = bx * bx;
    // total pressure, energy and fast magnetosonic speed of a side
    struct Side {
        double pt, e, cf;
    };
    auto side = [&](const double *w) {
        Side s;
        const double b1 = w[BCC + 1] * w[BCC + 1], b2 = w[BCC + 2] * w[BCC + 2];
        double pm = bx2 / 2;
        pm += b1 / 2;
        pm += b2 / 2;
        const double v2 = w[MOM] * w[MOM] + w[MOM + 1] * w[MOM + 1] + w[MOM + 2] * w[MOM + 2];
        s.e = w[ENE] * k.cv + w[RHO] * v2 / 2;
        s.e += pm;
        s.pt = w[ENE] + pm;
        const Den64 rho = den64(w[RHO]);
        const double cs2 = over64(w[ENE] * k.ge, rho);
        const double va2 = over64(bx2, rho);
        const double vt2 = over64(b1 + b2, rho);
        const double q2 = va2 + vt2 + cs2, r2 = va2 + vt2 - cs2;
        s.cf = ksqrt(0.5 * (q2 + ksqrt(r2 * r2 + 4 * cs2 * vt2)));
        return s;
    };
    const Side l = side(wl), r = side(wr);
    const double ul = wl[MOM], ur = wr[MOM];
    const double sm2 = vmin(ul - l.cf, ur - r.cf), sp2 = vmax(ul + l.cf, ur + r.cf);
    const bool super_ = sm2 >= 0 || sp2 <= 0;
    const double sdl = sm2 - ul, sdr = sp2 - ur;
    const double ml = wl[RHO] * ul, mr = wr[RHO] * ur;
    const double s0 = over64(sdr * mr - r.pt - sdl * ml + l.pt, den64(sdr * wr[RHO] - sdl * wl[RHO]));
    const double sdml = sm2 - s0, sdmr = sp2 - s0;
    const Den64 dsml = den64(sdml), dsmr = den64(sdmr);
    const double rsdl = wl[RHO] * sdl, rsdr = wr[RHO] * sdr;
    const double rl = over64(rsdl, dsml), rr = over64(rsdr, dsmr);       // rho*
    const double ql = ksqrt(rl), qr = ksqrt(rr);
    const Den64 dql = den64(ql), dqr = den64(qr);
    const double abx = vabs(bx);
    const double sm1 = s0 - over64(abx, dql), sp1 = s0 + over64(abx, dqr);
    const double tiny = (double)(1.00e-4f);
    const double pts = l.pt + rsdl * (sdl - sdml);
    struct Star {
        double m1, m2, b1, b2;
    };
    auto star = [&](const double *w, double rsd, double sd, double sdm, double rs) {
        Star o;
        const double dn = rsd * sdm - bx2;
        const bool deg = vabs(dn) < tiny * pts;
        const Den64 dd = den64(dn);
        const double tv = over64(bx * (sd - sdm), dd), tb = over64(rsd * sd - bx2, dd);
        o.m1 = rs * sel(deg, w[MOM + 1], w[MOM + 1] - w[BCC + 1] * tv);
        o.m2 = rs * sel(deg, w[MOM + 2], w[MOM + 2] - w[BCC + 2] * tv);
        o.b1 = sel(deg, w[BCC + 1], w[BCC + 1] * tb);
        o.b2 = sel(deg, w[BCC + 2], w[BCC + 2] * tb);
        return o;
    };
    const Star L = star(wl, rsdl, sdl, sdml, rl), R = star(wr, rsdr, sdr, sdmr, rr);

    // double-star transverse velocities and fields (hlld.h:246-276)
    const bool dbl = bx2 > pts * tiny;
    const double sg = bx > 0 ? 1.0 : -1.0;
    const Den64 drl = den64(rl), drr = den64(rr);
    const double inv = over64(1.0, den64(ql + qr));
    const double sq = sg * ql * qr;
    const double v1 = inv * (over64(L.m1, dql) + over64(R.m1, dqr) + sg * (R.b1 - L.b1));
    const double v2 = inv * (over64(L.m2, dql) + over64(R.m2, dqr) + sg * (R.b2 - L.b2));
    const double c1 = inv * (ql * R.b1 + qr * L.b1 + sq * (over64(R.m1, drr) - over64(L.m1, drl)));
    const double c2 = inv * (ql * R.b2 + qr * L.b2 + sq * (over64(R.m2, drr) - over64(L.m2, drl)));
    const double te = s0 * bx + over64(rl * v1 * c1 + rl * v2 * c2, drl);

    // the side of the contact that the flux takes
    const bool star1 = sm1 >= 0, star2 = !star1 && sp1 <= 0;
    const bool left = super_ ? sm2 >= 0 : (star1 || (!star2 && s0 >= 0));
    const double rho = sel(left, wl[RHO], wr[RHO]), u = sel(left, ul, ur);
    const double w1 = sel(left, wl[MOM + 1], wr[MOM + 1]), w2 = sel(left, wl[MOM + 2], wr[MOM + 2]);
    const double b1 = sel(left, wl[BCC + 1], wr[BCC + 1]), b2 = sel(left, wl[BCC + 2], wr[BCC + 2]);
    const double e = sel(left, l.e, r.e), pt = sel(left, l.pt, r.pt);
    const double sd = sel(left, sdl, sdr), rs = sel(left, rl, rr), q = sel(left, ql, qr);
    const double a2 = sel(left, sm2, sp2), a1 = sel(left, sm1, sp1);
    const Den64 dsm = {sel(left, dsml.d, dsmr.d), sel(left, dsml.r, dsmr.r)};
    const Den64 drs = {rs, sel(left, drl.r, drr.r)};
    const Star S = {sel(left, L.m1, R.m1), sel(left, L.m2, R.m2), sel(left, L.b1, R.b1), sel(left, L.b2, R.b2)};
    const double m = rho * u, m1 = rho * w1, m2 = rho * w2, ms = rs * s0;
    // star energy (hlld.h:192-200), double-star energy
    const double udb = over64(ms * bx + S.m1 * S.b1 + S.m2 * S.b2, drs);
    const double wdb = u * bx + w1 * b1 + w2 * b2;
    const double es = over64(bx * (wdb - udb) - pt * u + sd * e + pts * s0, dsm);
    const double de = q * sg * (udb - te);
    const double ess = left ? es - de : es + de;
    const double x1 = sel(dbl, rs * v1, S.m1), x2 = sel(dbl, rs * v2, S.m2);
    const double y1 = sel(dbl, c1, S.b1), y2 = sel(dbl, c2, S.b2), xe = sel(dbl, ess, es);
    // physical flux of the side (hlld.h:49-69)
    const double f0 = m, fe = u * (pt + e - bx2) - bx * (w1 * b1 + w2 * b2), fm = pt - bx2 + m * u;
    const double f1 = -bx * b1 + m1 * u, f2 = -bx * b2 + m2 * u;
    const double g1 = -bx * w1 + b1 * u, g2 = -bx * w2 + b2 * u;
    const bool one = star1 || star2;
    const double dv = a1 - a2;
    auto fan = [&](double f, double uu, double us, double uss) {
        const double s = f + a2 * (us - uu);
        const double d = f + (-a2 * uu - dv * us + a1 * uss);
        return sel(super_, f, sel(one, s, d));
    };
    flx[RHO] = fan(f0, rho, rs, rs);
    flx[ENE] = fan(fe, e, es, xe);
    flx[MOM] = fan(fm, m, ms, ms);
    flx[MOM + 1] = fan(f1, m1, S.m1, x1);
    flx[MOM + 2] = fan(f2, m2, S.m2, x2);
    flx[BCC] = 0;
    flx[BCC + 1] = fan(g1, b1, S.b1, y1);
    flx[BCC + 2] = fan(g2, b2, S.b2, y2);
}

// hllc<double> (hydro/riemann/hllc.h:76-193): 10 quotients over 8
// denominators, fluxes of the upwind side only (the other side's weight is
// 0).  Its guard for products past FLT_MAX / 10 and for a vanishing mass sum
// are the general function's, as are inputs out of range.
__device__ __forceinline__ void hllc64(double *flx, const double *wl, const double *wr, const Gam64 &k) {
    struct Side {
        double e, c, q;          // total energy, sound speed, sqrt(rho)
    };
    auto side = [&](const double *w) {
        Side s;
        const double v2 = w[MOM] * w[MOM] + w[MOM + 1] * w[MOM + 1] + w[MOM + 2] * w[MOM + 2];
        s.e = w[ENE] * k.cv + w[RHO] * v2 / 2;
        s.c = ksqrt(k.g * over64(w[ENE], den64(w[RHO])));
        s.q = ksqrt(w[RHO]);
        return s;
    };
    const Side l = side(wl), r = side(wr);
    const double isd = over64(1.0, den64(l.q + r.q));
    double v[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) v[n] = (l.q * wl[MOM + n] + r.q * wr[MOM + n]) * isd;
    const double h = isd * (over64(l.e + wl[ENE], den64(l.q)) + over64(r.e + wr[ENE], den64(r.q)));
    const double g1 = over64(1.0, den64(isd * (l.q * k.cv + r.q * k.cv)));
    const double q = h - 0.5 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    const double a = q <= 0 ? 0.0 : ksqrt(g1 * q);
    const double al = pmin(v[0] - a, wl[MOM] - l.c), ar = pmax(v[0] + a, wr[MOM] + r.c);
    const double bp = ar > 0 ? ar : 0.0, bm = al < 0 ? al : 0.0;
    const double vxl = wl[MOM] - al, vxr = wr[MOM] - ar;
    const double tl = wl[ENE] + vxl * wl[RHO] * wl[MOM], tr = wr[ENE] + vxr * wr[RHO] * wr[MOM];
    const double ml = wl[RHO] * vxl, mr = -wr[RHO] * vxr;
    {
        const double lo = 0x1p-60;
        const double p1 = ml * tr, p2 = mr * tl;
        const bool in = kfabs(p1) + kfabs(p2) + l.e + r.e + wl[RHO] + wr[RHO] < 0x1p60 && ml + mr > lo &&
                        wl[RHO] > lo && wr[RHO] > lo && wl[ENE] > lo && wr[ENE] > lo;
        if (__builtin_expect(!__all(in), 0)) {
            hllc<double>(flx, wl, wr, k.g);
            return;
        }
    }
    const Den64 ms = den64(ml + mr);
    const double am = over64(tl - tr, ms);
    const double cp = pmax(over64(ml * tr + mr * tl, ms), 0.0);
    const bool left = am >= 0;
    const double b = am > 0 ? bm : bp, bx = left ? bm : bp;
    const double f_min = (double)(FLT_MIN * 1e1f);
    const Den64 d = den64(pmax(kfabs(am - b), f_min) * (am > b ? 1 : -1));
    const double s = over64(am, d), sm = over64(-b, d);
    const double rho = sel(left, wl[RHO], wr[RHO]), p = sel(left, wl[ENE], wr[ENE]);
    const double u = sel(left, wl[MOM], wr[MOM]), e = sel(left, l.e, r.e);
    const double vn = u - bx;
    flx[RHO] = s * (rho * vn);
    flx[ENE] = s * (p * u + e * vn);
    flx[MOM] = s * (rho * u * vn + p);
    flx[MOM + 1] = s * (rho * sel(left, wl[MOM + 1], wr[MOM + 1]) * vn);
    flx[MOM + 2] = s * (rho * sel(left, wl[MOM + 2], wr[MOM + 2]) * vn);
    flx[MOM] += sm * cp;
    flx[ENE] += sm * cp * am;
}

// Face flux in the mesh frame for a sweep along `axis`: hllc.h:32-43 and
// hlld.h:29-47 (the B-flux slots are rewritten as edge EMFs, normal slot 0).
// ql / qr are rotated in place.
template <class FT, bool MHD, int AXIS>
__device__ __forceinline__ void face_flux(FT *ql, FT *qr, FT *flx, const Gam64 &k) {
    rot<AXIS>(ql + MOM);
    rot<AXIS>(qr + MOM);
    if constexpr (MHD) {
        rot<AXIS>(ql + BCC);
        rot<AXIS>(qr + BCC);
        if constexpr (std::is_same_v<FT, float>)
            hlld_fast(flx, ql, qr, (float)k.g);
        else
            hlld64(flx, ql, qr, k);
        rot<3 - AXIS>(flx + MOM);
        const FT e0 = flx[BCC + 2], e1 = -flx[BCC + 1];
        flx[BCC + (AXIS + 1) % 3] = e0;
        flx[BCC + (AXIS + 2) % 3] = e1;
        flx[BCC + AXIS] = 0;
    } else {
        if constexpr (std::is_same_v<FT, float>)
            hllc_fast(flx, ql, qr, (float)k.g);
        else
            hllc64(flx, ql, qr, k);
        rot<3 - AXIS>(flx + MOM);
    }
}

}  // namespace kr
