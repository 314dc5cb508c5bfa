// pk_adjoint.hpp -- reverse mode (vector-Jacobian products) of the per-cell
// and per-interface arithmetic of the hydro sweep in pk_math.hpp:
//   prim_vjp_hd()   utoq            (interpolations.F90:69-106)
//   limit_vjp()     the limiters    (fluxlimiters.F90:109-216)
//   hllc_vjp()      riemann_hlld_u  (hlld.F90:615-841)
//   hlld_vjp()      riemann_hlld with the GLM psi flux (hlld.F90:161-609)
//   prim_vjp_mhd()  utoq with B
//   floors_vjp_hd(), floors_vjp_mhd()   care_for_positives (sources.F90:299-433)
//   dt_vjp_hd(), dt_vjp_mhd()           timestep_fluid at one cell
//                   (timestep.F90:460-490 with neu_cs / ion_cs)
//
// Each function re-evaluates the forward values that select a branch (wave
// speeds and their signs, the star-state tests, limiter cases, min/max
// choices, floors) in the forward's order with the forward's bits (ndiv and
// nsqrt: those of the exact division and square root for operands away from
// the ends of the exponent range, and their special values), and then runs the chain rule backwards
// through the branch the forward took.  Quotients that only scale adjoints
// are formed with one reciprocal per divisor: they differ from a division by
// at most an ulp, far below the derivative's own truncation, and an IEEE
// division costs about ten FP64 instructions.
// Where a min or max has two exactly equal arguments the derivative is split
// evenly between them (the forward value does not depend on the choice).
#pragma once
#include "pk_math.hpp"

namespace PK_KNS {

// x, unknown to the compiler from here on (device): values derived from it
// before and after are formed twice instead of being held in registers in
// between, which the long reverse passes need to fit two waves per SIMD.
PK_HD void forget(double &x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
}

// x with its sign changed unless keep.
PK_HD double signed_(bool keep, double x) { return keep ? x : -x; }

// d min(a, b): weights of a and b
PK_HD void dmin(double a, double b, double &wa, double &wb)
{
    wa = (a < b) ? 1.0 : ((a > b) ? 0.0 : 0.5);
    wb = 1.0 - wa;
}
PK_HD void dmax(double a, double b, double &wa, double &wb)
{
    wa = (a > b) ? 1.0 : ((a < b) ? 0.0 : 0.5);
    wb = 1.0 - wa;
}

PK_HD void swap_(double &a, double &b)
{
    const double t = a;
    a = b;
    b = t;
}

// ---- utoq (HD) -------------------------------------------------------------
// q = prim(u); given qb = dL/dq, add dL/du to ub.
PK_HD void prim_vjp_hd(const double (&u)[5], double gam_1, const double (&qb)[5], double (&ub)[5])
{
    const double rd = nrcp(u[0]);
    const double q1 = u[1] * rd, q2 = u[2] * rd, q3 = u[3] * rd;
    const double ek = (0.5 * ((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3])) * rd;
    // p = gam_1 * (E - ek)
    double db = qb[0];
    ub[4] += gam_1 * qb[4];
    const double ekb = -(gam_1 * qb[4]);
    // ek = S / d, S = 0.5*(m1^2 + m2^2 + m3^2)
    const double sb = ekb * rd;
    db -= sb * ek;
    ub[1] += sb * u[1];
    ub[2] += sb * u[2];
    ub[3] += sb * u[3];
    // v_k = m_k / d
    ub[1] += qb[1] * rd;
    ub[2] += qb[2] * rd;
    ub[3] += qb[3] * rd;
    db -= (qb[1] * q1 + qb[2] * q2 + qb[3] * q3) * rd;
    ub[0] += db;
}

// ---- limiters ----------------------------------------------------------------
// dq = limit(lim, dl, dr); given dqb, return dL/d(dl), dL/d(dr).
PK_HD void limit_vjp(int lim, double dl, double dr, double dqb, double &dlb, double &drb)
{
    dlb = 0.0;
    drb = 0.0;
    if (lim == LIM_VANLEER) {
        const double dcen = dl * dr;
        if (dcen > 0.0) {
            // 2*dl*dr/(dl+dr); the quotients are at most 1 each, where the square
            // of the reciprocal overflows for slopes below 1e-154
            const double rs = nrcp(dl + dr), x = dr * rs, y = dl * rs, g = 2.0 * dqb;
            dlb = g * (x * x);
            drb = g * (y * y);
        }
        return;
    }
    const double sgl = copysign(1.0, dl), sgr = copysign(1.0, dr);
    const double s = sgl + sgr;
    if (s == 0.0) return;  // opposite signs: zero slope
    const double a = fabs(dl), b = fabs(dr);
    if (lim == LIM_MINMOD) {
        // (s * min(a, b)) * 0.5
        double wa, wb;
        dmin(a, b, wa, wb);
        const double mb = (s * 0.5) * dqb;
        dlb = mb * wa * sgl;
        drb = mb * wb * sgr;
        return;
    }
    if (lim == LIM_MONCEN) {
        // (s * min(min(2a, 2b), 0.5*|dl+dr|)) * 0.5
        const double m1 = fmn(2.0 * a, 2.0 * b), m2 = 0.5 * fabs(dl + dr);
        double w1, w2, wa, wb;
        dmin(m1, m2, w1, w2);
        dmin(2.0 * a, 2.0 * b, wa, wb);
        const double mb = (s * 0.5) * dqb;
        const double sc = copysign(1.0, dl + dr);
        dlb = mb * (w1 * wa * 2.0 * sgl + w2 * 0.5 * sc);
        drb = mb * (w1 * wb * 2.0 * sgr + w2 * 0.5 * sc);
        return;
    }
    // superbee: (s*0.5) * (a > b ? min(a, |2 dr|) : min(|2 dl|, b))
    const double mb = (s * 0.5) * dqb;
    double w1, w2;
    if (a > b) {
        dmin(a, fabs(2.0 * dr), w1, w2);
        dlb = mb * w1 * sgl;
        drb = mb * w2 * 2.0 * sgr;
    } else {
        dmin(fabs(2.0 * dl), b, w1, w2);
        dlb = mb * w1 * 2.0 * sgl;
        drb = mb * w2 * sgr;
    }
}

// ---- HLLC and HLLD ---------------------------------------------------------------
//
// Both solvers return the flux of one side of the contact: the upwind side
// when the flow is supersonic, else the side sm > 0 names (left) -- every
// region test of the forward solver (Alfven speeds included) selects the
// side the contact speed points to -- and the average of the two sides when
// sm == 0.  The reverse pass is written once, for side A = the selected side
// and side O = the other one, with sg = +1 when A is the left side; the two
// sides' formulas are mirror images.  In the averaged case both sides count
// with weight 1/2 (the pass is linear in the flux adjoint given the branch):
// HLLC adds O's own part to A's and runs what they share (sm, the star
// pressure, the wave speeds) once, HLLD runs its pass twice.  Isobaric gas at
// rest averages at every interface: a 128^3 hydro reverse sweep along x, y, z
// takes 222, 211, 209 us there and 229, 226, 225 in moving gas; with HLLC's
// pass run twice, its first result in scratch memory, 345, 388, 390 at rest.

// The flux of side A and its reverse, shared by both solvers: with
// dn = q0*(s - q1) and ds = dn/(s - sm) the side's star flux F + s*(U* - U) is
//   [s*ds - dn, pt - dn*q1 + s*ds*sm, s*ds*vy - dn*q2, s*ds*vz - dn*q3,
//    pt*q1 - x*en + s*us4], x = s - q1
// (B terms apart), which needs neither F nor U.

// Adjoints of what a side's star flux takes from the interface.
struct HllcSide {
    double ssm, x, p, prt, sm, dn, s;
};

// f = flux_hllc(l, r); given fb, add dL/dl to lb and dL/dr to rb.
// rg1 = 1/(gam - 1).
PK_HD void hllc_vjp_r(const double *l, const double *r, double gam, double rg1, const double *fb, double *lb,
                      double *rb)
{
    const double cl2 = ndiv(gam * l[4], l[0], nrcp(l[0])), cr2 = ndiv(gam * r[4], r[0], nrcp(r[0]));
    const double c = nsqrt(fmx(cl2, cr2));
    const double sl = fmn(l[1], r[1]) - c;
    const double sr = fmx(l[1], r[1]) + c;
    if (sl >= 0.0 || sr <= 0.0) {
        // the upwind physical flux
        const bool L = sl >= 0.0;
        double q[5], o[5];
#pragma unroll
        for (int v = 0; v < 5; v++) q[v] = L ? l[v] : r[v];
        const double K = (q[1] * q[1] + q[2] * q[2]) + q[3] * q[3];
        const double en = (q[4] * rg1) + (0.5 * q[0]) * K;
        const double W = fb[0] + fb[1] * q[1] + fb[2] * q[2] + fb[3] * q[3];  // adjoint of q0*q1
        const double m = q[0] * q[1];
        const double enb = fb[4] * q[1];
        const double kb = enb * q[0];
        o[0] = W * q[1] + (0.5 * enb) * K;
        o[1] = W * q[0] + fb[1] * m + fb[4] * (en + q[4]) + kb * q[1];
        o[2] = fb[2] * m + kb * q[2];
        o[3] = fb[3] * m + kb * q[3];
        o[4] = fb[1] + enb + enb * rg1;
#pragma unroll
        for (int v = 0; v < 5; v++) {
            lb[v] += L ? o[v] : 0.0;
            rb[v] += L ? 0.0 : o[v];
        }
        return;
    }
    const double auxr = (sr - r[1]) * r[0], auxl = (sl - l[1]) * l[0];
    const bool degen = fabs(auxr - auxl) < spacing(auxr + auxl);
    const double rden = nrcp(auxr - auxl);
    const double sm = degen ? (sl + sr) / 2.0
                            : ndiv((auxr * r[1] - r[4]) - (auxl * l[1] - l[4]), auxr - auxl, rden);
    const double prt = 0.5 * ((l[4] + auxl * (sm - l[1])) + (r[4] + auxr * (sm - r[1])));
    const bool both = sm == 0.0, left = sm > 0.0;
    const double w = both ? 0.5 : 1.0;
    double a[5], o[5], ab[5], ob[5];
#pragma unroll
    for (int v = 0; v < 5; v++) {
        a[v] = left ? l[v] : r[v];
        o[v] = left ? r[v] : l[v];
    }
    const double s = left ? sl : sr, so = left ? sr : sl;
    const double ca2 = left ? cl2 : cr2, co2 = left ? cr2 : cl2;
    const double rdo = left ? rden : -rden;  // 1/(dno - dn)
    const double x = s - a[1], xo = so - o[1];
    const double dn = a[0] * x, dno = o[0] * xo;
    // the side's own part: from the flux adjoint to those of its state and of
    // what both sides share (x = s - q1, dn, en, prt, sm, s - sm)
    auto side = [&](const double (&q)[5], double s_, double x_, double dn_, double (&qb)[5], HllcSide &y) {
        const double K = (q[1] * q[1] + q[2] * q[2]) + q[3] * q[3];
        const double en = (q[4] * rg1) + (0.5 * q[0]) * K;
        const double rs = nrcp(s_ - sm);
        const double d = dn_ * rs;
        const double us4 = (((x_ * en) - (q[4] * q[1])) + (prt * sm)) * rs;
        const double g0 = w * fb[0], g1 = w * fb[1], g2 = w * fb[2], g3 = w * fb[3], g4 = w * fb[4];
        const double sd = s_ * d, W = sd - dn_;
        const double Wb = (g0 + g2 * q[2]) + g3 * q[3];
        const double sdb = Wb + g1 * sm;
        const double nb = (g4 * s_) * rs;
        const double dr = (sdb * s_) * rs;
        y.ssm = -(nb * us4) - dr * d;
        y.x = nb * en - g4 * en;
        const double enb = nb * x_ - g4 * x_;
        const double pf = g4 - nb;  // pt*q1 - (pt*q1 in the star energy)
        y.p = g1 + pf * q[1];
        y.prt = nb * sm;
        y.sm = g1 * sd + nb * prt;
        y.dn = dr - Wb - g1 * q[1];
        const double kb = enb * q[0];
        qb[0] = (0.5 * enb) * K;
        qb[1] = kb * q[1] - g1 * dn_ + pf * q[4];
        qb[2] = g2 * W + kb * q[2];
        qb[3] = g3 * W + kb * q[3];
        qb[4] = enb * rg1;
        y.s = sdb * d + g4 * us4 + y.ssm;
    };
    HllcSide y, yo;
    side(a, s, x, dn, ab, y);
    yo.ssm = yo.x = yo.p = yo.prt = yo.sm = yo.dn = yo.s = 0.0;
#pragma unroll
    for (int v = 0; v < 5; v++) ob[v] = 0.0;
    if (both) side(o, so, xo, dno, ob, yo);
    const double h = 0.5 * (y.prt + yo.prt);
    const double smb = (y.sm + yo.sm) + h * (dn + dno) - y.ssm - yo.ssm;
    double dnb = y.dn + h * (sm - a[1]), dnob = yo.dn + h * (sm - o[1]);
    double sb = y.s, sob = yo.s;
    ab[1] -= h * dn;
    ob[1] -= h * dno;
    double pb = y.p + h, pob = yo.p + h;
    // sm = ((dno*o1 - po) - (dn*a1 - pa)) / (dno - dn), or the mirror image of it
    if (degen) {
        sb += 0.5 * smb;
        sob += 0.5 * smb;
    } else {
        const double q = smb * rdo;
        dnob += q * (o[1] - sm);
        dnb -= q * (a[1] - sm);
        ob[1] += q * dno;
        ab[1] -= q * dn;
        pob -= q;
        pb += q;
    }
    // dn = q0*x, x = s - q1
    ab[0] += dnb * x;
    const double xb = y.x + dnb * a[0];
    ob[0] += dnob * xo;
    const double xob = yo.x + dnob * o[0];
    sb += xb;
    ab[1] -= xb;
    sob += xob;
    ob[1] -= xob;
    ab[4] += pb;
    ob[4] += pob;
    // sl = min(l1, r1) - c, sr = max(l1, r1) + c, c = sqrt(max(cl2, cr2))
    const double lowb = left ? sb : sob, highb = left ? sob : sb;
    double wa, wo;
    dmin(a[1], o[1], wa, wo);
    ab[1] += lowb * wa;
    ob[1] += lowb * wo;
    dmax(a[1], o[1], wa, wo);
    ab[1] += highb * wa;
    ob[1] += highb * wo;
    const double cmb = (highb - lowb) * (0.5 * nrcp(c));
    dmax(ca2, co2, wa, wo);
    const double ga = (cmb * wa) * nrcp(a[0]), go = (cmb * wo) * nrcp(o[0]);
    ab[4] += ga * gam;
    ab[0] -= ga * ca2;
    ob[4] += go * gam;
    ob[0] -= go * co2;
#pragma unroll
    for (int v = 0; v < 5; v++) {
        lb[v] += left ? ab[v] : ob[v];
        rb[v] += left ? ob[v] : ab[v];
    }
}

PK_HD void hllc_vjp(const double *l, const double *r, double gam, const double *fb, double *lb, double *rb)
{
    hllc_vjp_r(l, r, gam, 1.0 / (gam - 1.0), fb, lb, rb);
}

// ---- HLLD + GLM ----------------------------------------------------------------

// f = flux_hlld(l, r, gam, ch); given fb[9], add dL/dl to lb, dL/dr to rb
// and return dL/dch.  rg = 1/gam, rg1 = 1/(gam - 1), rch = 1/ch.
PK_HD double hlld_vjp_r(const double *l, const double *r, double gam, double rg, double rg1, double ch, double rch,
                        const double *fb, double *lb, double *rb)
{
    // GLM fluxes (hlld.F90:229-230)
    const double kch = (ch * ch) * 0.5;
    const double A = (r[5] + l[5]) - (r[8] - l[8]) * rch;
    const double chb = fb[8] * (ch * A + 0.5 * (r[8] - l[8])) - fb[5] * 0.5 * (r[5] - l[5]);
    lb[5] += fb[8] * kch + fb[5] * 0.5 * ch;
    rb[5] += fb[8] * kch - fb[5] * 0.5 * ch;
    const double g8 = fb[8] * kch * rch;
    lb[8] += g8 + fb[5] * 0.5;
    rb[8] += -g8 + fb[5] * 0.5;

    // ---- forward values of both sides ----
    const double b2l = (l[5] * l[5] + l[6] * l[6]) + l[7] * l[7];
    const double b2r = (r[5] * r[5] + r[6] * r[6]) + r[7] * r[7];
    const double prl = l[4] + 0.5 * b2l;
    const double prr = r[4] + 0.5 * b2r;
    const double gpl = gam * l[4], gpr = gam * r[4];
    const double tl = gpl + b2l, tr = gpr + b2r;
    const double sql = nsqrt(tl * tl - (4.0 * gpl) * (l[5] * l[5]));
    const double sqr = nsqrt(tr * tr - (4.0 * gpr) * (r[5] * r[5]));
    const double cl = ndiv(tl + sql, l[0], nrcp(l[0]));
    const double cr = ndiv(tr + sqr, r[0], nrcp(r[0]));
    const double c = nsqrt(0.5 * fmx(cl, cr));
    const double sl = fmn(l[1], r[1]) - c;
    const double sr = fmx(l[1], r[1]) + c;

    if (sl >= 0.0 || sr <= 0.0) {
        // the upwind physical flux: pt = p + b2/2, en = p/(gam-1) + q0*K/2 + b2/2, W = v.B
        const bool L = sl >= 0.0;
        double q[8], o[8];
#pragma unroll
        for (int v = 0; v < 8; v++) q[v] = L ? l[v] : r[v];
        const double b2 = L ? b2l : b2r, pt = L ? prl : prr;
        const double K = (q[1] * q[1] + q[2] * q[2]) + q[3] * q[3];
        const double en = ((q[4] * rg1) + (0.5 * q[0]) * K) + 0.5 * b2;
        const double W = (q[1] * q[5] + q[2] * q[6]) + q[3] * q[7];
        const double m = q[0] * q[1];
        const double mb = fb[0] + fb[1] * q[1] + fb[2] * q[2] + fb[3] * q[3];
        const double enb = fb[4] * q[1];
        const double kb = enb * q[0];
        const double ptb = fb[1] + enb;
        const double Wb = -(fb[4] * q[5]);
        const double b2b = enb + ptb;  // twice d/d(b2): the factors 2*B below are halved
        o[0] = mb * q[1] + (0.5 * enb) * K;
        o[1] = mb * q[0] + fb[1] * m + fb[4] * (en + pt) + kb * q[1] + Wb * q[5] + fb[6] * q[6] + fb[7] * q[7];
        o[2] = fb[2] * m + kb * q[2] + Wb * q[6] - fb[6] * q[5];
        o[3] = fb[3] * m + kb * q[3] + Wb * q[7] - fb[7] * q[5];
        o[4] = ptb + enb * rg1;
        o[5] = Wb * q[1] - fb[4] * W - 2.0 * q[5] * fb[1] - q[6] * fb[2] - q[7] * fb[3] - fb[6] * q[2] -
               fb[7] * q[3] + b2b * q[5];
        o[6] = Wb * q[2] - q[5] * fb[2] + fb[6] * q[1] + b2b * q[6];
        o[7] = Wb * q[3] - q[5] * fb[3] + fb[7] * q[1] + b2b * q[7];
#pragma unroll
        for (int v = 0; v < 8; v++) {
            lb[v] += L ? o[v] : 0.0;
            rb[v] += L ? 0.0 : o[v];
        }
        return chb;
    }

    double sm;
    bool degen;
    {
        const double auxr = (sr - r[1]) * r[0], auxl = (sl - l[1]) * l[0];
        degen = fabs(auxr - auxl) < spacing(auxr + auxl);
        sm = degen ? (sl + sr) / 2.0
                   : ndiv((auxr * r[1] - prr) - (auxl * l[1] - prl), auxr - auxl, nrcp(auxr - auxl));
    }
    const bool both = sm == 0.0;
    bool left = sm > 0.0;
    const bool bxnz = fabs(l[5]) > 0.0, bpos = l[5] >= 0.0;
    // which side's speed the maximum is (cl == cr: both, half each)
    const bool maxl = cl >= cr, maxr = cr >= cl;
    // ---- side A and the other side O ----
    double a[8], o[8], ab[8], ob[8];
    volatile double first[16];  // the first pass of an averaged interface (rare: kept out of registers)
#pragma unroll
    for (int v = 0; v < 8; v++) {
        a[v] = left ? l[v] : r[v];
        o[v] = left ? r[v] : l[v];
    }
    double s = left ? sl : sr, so = left ? sr : sl, cc = c;
    for (int pass = 0;; pass++) {
        double sb, sob = 0.0, smb, dnb, dnob = 0.0, xob = 0.0, ssmb, ssmob = 0.0, xb, ptb, prtb, enb, bbb = 0.0;
        double hyb = 0.0, hzb = 0.0;
        bool hll, oka;
        {
            const double bb = a[5] * o[5];
            const double bbg = ndiv(bb, gam, rg);
            const double bmin = spacing(bb);
            const double x = s - a[1];
            const double dn = a[0] * x;
            const double ssm = s - sm;
            const double rs = nrcp(ssm);
            const double ds = ndiv(dn, ssm, rs);
            const double c1 = dn * ssm - bb;
            oka = (fabs(c1) > bmin) && bbg <= a[4];
            const double xo = so - o[1];
            const double dno = o[0] * xo;
            const double ssmo = so - sm;
            const double c2 = dno * ssmo - bb;
            const bool oko = (fabs(c2) > bmin) && bbg <= o[4];
            hll = !(oka && oko);
            double hy = 0.0, hz = 0.0;
            if (hll) {
                const double rh = nrcp(so - s);
                hy = ((so * o[6] - s * a[6]) - ((o[6] * o[1] - o[5] * o[2]) - (a[6] * a[1] - a[5] * a[2]))) * rh;
                hz = ((so * o[7] - s * a[7]) - ((o[7] * o[1] - o[5] * o[3]) - (a[7] * a[1] - a[5] * a[3]))) * rh;
            }
            const double r1 = nrcp(c1);
            const double t1 = (dn * x - bb) * r1;
            const double by = oka ? a[6] * t1 : hy, bz = oka ? a[7] * t1 : hz;
            const double rdn = nrcp(dn);
            const double ol = a[5] * rdn;
            const double vy = a[2] + ol * (a[6] - by), vz = a[3] + ol * (a[7] - bz);
            const double sq = nsqrt(ds), rq = nrcp(sq);
            const double al = sm - signed_(left, ndiv(fabs(a[5]), sq, rq));
            // between the Alfven waves: the double-star state (hlld.F90:458-474)
            const bool dbl = bxnz && (left ? !(al > 0.0) : !(al < 0.0));
            const double vbs = (sm * a[5] + vy * by) + vz * bz;

            // ---- reverse of the side's star flux ----
            //   f0 = s*ds - dn, f1 = pt - dn*q1 - q5^2 + s*ds*sm, f2 = s*ds*vy - dn*q2 - q5*q6,
            //   f4 = pt*q1 - x*en - q5*vb + s*us4, f6 = s*by - x*q6 - q5*q2 (f3, f7 alike), and
            //   in the double-star region + al*(U** - U*)
            double g[8];
#pragma unroll
            for (int v = 0; v < 8; v++) g[v] = both ? 0.5 * fb[v] : fb[v];
            double dsb, vyb, vzb, byb, bzb, vbsb;
            {
                const double b2 = (a[5] * a[5] + a[6] * a[6]) + a[7] * a[7];
                const double pt = a[4] + 0.5 * b2;
                const double pto = o[4] + 0.5 * ((o[5] * o[5] + o[6] * o[6]) + o[7] * o[7]);
                const double prt = 0.5 * ((pt + dn * (sm - a[1])) + (pto + dno * (sm - o[1])));
                const double K = (a[1] * a[1] + a[2] * a[2]) + a[3] * a[3];
                const double en = ((a[4] * rg1) + (0.5 * a[0]) * K) + 0.5 * b2;
                const double vb = (a[1] * a[5] + a[2] * a[6]) + a[3] * a[7];
                const double us4 = ((((x * en) - (pt * a[1])) + (prt * sm)) + a[5] * (vb - vbs)) * rs;
                const double sd = s * ds;
                const double sdb = ((g[0] + g[1] * sm) + g[2] * vy) + g[3] * vz;
                sb = sdb * ds + (g[4] * us4 + g[6] * by) + g[7] * bz;
                dsb = sdb * s;
                smb = g[1] * sd;
                vyb = g[2] * sd;
                vzb = g[3] * sd;
                dnb = -(((g[0] + g[1] * a[1]) + g[2] * a[2]) + g[3] * a[3]);
                byb = s * g[6];
                bzb = s * g[7];
                // us4 = n/ssm, n = ((x*en - pt*q1) + prt*sm) + q5*(vb - vbs)
                const double nb = (s * g[4]) * rs;
                ssmb = -(nb * us4);
                const double nf = nb - g[4];
                enb = nf * x;
                xb = (nf * en - g[6] * a[6]) - g[7] * a[7];
                ptb = g[1] - nf * a[1];
                prtb = nb * sm;
                smb += nb * prt;
                const double vbb = nf * a[5];
                vbsb = -(nb * a[5]);
                const double kb = enb * a[0];
                ab[1] = kb * a[1] + vbb * a[5] - g[1] * dn - nf * pt;
                ab[2] = kb * a[2] + vbb * a[6] - g[2] * dn - g[6] * a[5];
                ab[3] = kb * a[3] + vbb * a[7] - g[3] * dn - g[7] * a[5];
                ab[5] = vbb * a[1] + nb * (vb - vbs) - g[4] * vb - 2.0 * a[5] * g[1] - g[2] * a[6] - g[3] * a[7] -
                        g[6] * a[2] - g[7] * a[3];
                ab[6] = vbb * a[2] - g[2] * a[5] - g[6] * x;
                ab[7] = vbb * a[3] - g[3] * a[5] - g[7] * x;
            }
            ob[1] = ob[2] = ob[3] = ob[5] = ob[6] = ob[7] = 0.0;
            forget(so);
            forget(s);
            if (dbl) {
                // ---- double star: needs the other side's star state ----
                const double xo2 = so - o[1];
                const double dno2 = o[0] * xo2;
                const double ssmo2 = so - sm;
                const double bb2 = a[5] * o[5];
                const double rso = nrcp(ssmo2);
                const double dso = dno2 * rso;
                const double sqo = nsqrt(dso);
                const double r2 = nrcp(dno2 * ssmo2 - bb2);
                const double t2 = (dno2 * xo2 - bb2) * r2;
                const double byo = oko ? o[6] * t2 : hy, bzo = oko ? o[7] * t2 : hz;
                const double rdno = nrcp(dno2);
                const double olo = o[5] * rdno;
                const double vyo = o[2] + olo * (o[6] - byo), vzo = o[3] + olo * (o[7] - bzo);
                const bool G = left == bpos;  // the sign of B_n as side A sees it
                const double radd = nrcp(sq + sqo);
                const double mul = sq * sqo;
                const double Gm = signed_(G, mul);
                const double v2y = ((sq * vy + sqo * vyo) + signed_(G, byo - by)) * radd;
                const double v2z = ((sq * vz + sqo * vzo) + signed_(G, bzo - bz)) * radd;
                const double b2y = ((sq * byo + sqo * by) + Gm * (vyo - vy)) * radd;
                const double b2z = ((sq * bzo + sqo * bz) + Gm * (vzo - vz)) * radd;
                const double b2x = 0.5 * (a[5] + o[5]);
                const double vb2 = (sm * b2x + v2y * b2y) + v2z * b2z;
                // + al*e: e2 = ds*(v2y - vy), e3 alike, e4 = -(G*sq)*(vbs - vb2), e6 = b2y - by, e7 alike
                const double dy = v2y - vy, dz = v2z - vz, dv = vbs - vb2, Gs = signed_(G, sq);
                const double alb =
                    (((g[2] * ds) * dy + (g[3] * ds) * dz) - (g[4] * Gs) * dv) + g[6] * (b2y - by) + g[7] * (b2z - bz);
                const double h2 = al * g[2], h3 = al * g[3], h4 = al * g[4], h6 = al * g[6], h7 = al * g[7];
                dsb += h2 * dy + h3 * dz;
                double v2yb = h2 * ds, v2zb = h3 * ds;
                vyb -= v2yb;
                vzb -= v2zb;
                double sqb = -(signed_(G, h4) * dv);
                const double u = Gs * h4;
                vbsb -= u;
                double b2yb = h6, b2zb = h7;
                byb -= h6;
                bzb -= h7;
                // vb2 = (sm*b2x + v2y*b2y) + v2z*b2z
                smb += u * b2x;
                const double hx = 0.5 * (u * sm);
                ab[5] += hx;
                ob[5] += hx;
                v2yb += u * b2y;
                b2yb += u * v2y;
                v2zb += u * b2z;
                b2zb += u * v2z;
                const double ny = b2yb * radd, nz = b2zb * radd, my = v2yb * radd, mz = v2zb * radd;
                const double addb = -(((ny * b2y + nz * b2z) + my * v2y) + mz * v2z);
                const double mulb = signed_(G, ny * (vyo - vy) + nz * (vzo - vz));
                sqb += (ny * byo + nz * bzo) + (my * vy + mz * vz) + addb + mulb * sqo;
                const double sqob = (ny * by + nz * bz) + (my * vyo + mz * vzo) + addb + mulb * sq;
                const double Gy = signed_(G, my), Gz = signed_(G, mz);
                byb += ny * sqo - Gy;
                bzb += nz * sqo - Gz;
                vyb += my * sq - ny * Gm;
                vzb += mz * sq - nz * Gm;
                const double vyob = ny * Gm + my * sqo, vzob = nz * Gm + mz * sqo;
                double byob = ny * sq + Gy, bzob = nz * sq + Gz;
                // al = sm - sg*|q5|/sq, sq = sqrt(ds)
                smb += alb;
                const double alq = signed_(left, alb * rq);
                ab[5] -= (a[5] > 0.0) ? alq : ((a[5] < 0.0) ? -alq : 0.0);
                sqb += (alq * rq) * fabs(a[5]);
                dsb += sqb * (0.5 * rq);
                // the other side: sqo = sqrt(dno/ssmo), vo = q + (q5/dn)*(q6 - byo), byo = q6*k/c2
                const double tt = (sqob * (0.5 * nrcp(sqo))) * rso;
                dnob += tt;
                ssmob -= tt * dso;
                ob[2] += vyob;
                ob[3] += vzob;
                const double olb = vyob * (o[6] - byo) + vzob * (o[7] - bzo);
                ob[6] += vyob * olo;
                byob -= vyob * olo;
                ob[7] += vzob * olo;
                bzob -= vzob * olo;
                ob[5] += olb * rdno;
                dnob -= (olb * olo) * rdno;
                if (oko) {
                    ob[6] += byob * t2;
                    ob[7] += bzob * t2;
                    const double kb2 = (byob * o[6] + bzob * o[7]) * r2;
                    const double c2b = -((byob * byo + bzob * bzo) * r2);
                    dnob += kb2 * xo2 + c2b * ssmo2;
                    xob += kb2 * dno2;
                    ssmob += c2b * dno2;
                    bbb -= kb2 + c2b;
                } else {
                    hyb += byob;
                    hzb += bzob;
                }
            }
            forget(s);
            // vbs = (sm*q5 + vy*by) + vz*bz
            smb += vbsb * a[5];
            ab[5] += vbsb * sm;
            vyb += vbsb * by;
            byb += vbsb * vy;
            vzb += vbsb * bz;
            bzb += vbsb * vz;
            // ds = dn/ssm
            const double dr = dsb * rs;
            dnb += dr;
            ssmb -= dr * ds;
            // v = q + (q5/dn)*(q6 - by)
            ab[2] += vyb;
            ab[3] += vzb;
            const double olb = vyb * (a[6] - by) + vzb * (a[7] - bz);
            ab[6] += vyb * ol;
            byb -= vyb * ol;
            ab[7] += vzb * ol;
            bzb -= vzb * ol;
            ab[5] += olb * rdn;
            dnb -= (olb * ol) * rdn;
            // by = q6*k1/c1, k1 = dn*x - bb, c1 = dn*ssm - bb
            if (oka) {
                const double x2 = s - a[1], dn2 = a[0] * x2;
                ab[6] += byb * t1;
                ab[7] += bzb * t1;
                const double kb1 = (byb * a[6] + bzb * a[7]) * r1;
                const double c1b = -((byb * by + bzb * bz) * r1);
                dnb += kb1 * x2 + c1b * (s - sm);
                xb += kb1 * dn2;
                ssmb += c1b * dn2;
                bbb -= kb1 + c1b;
            } else {
                hyb += byb;
                hzb += bzb;
            }
        }
        if (hll) {
            // h = ((so*o6 - s*a6) - (fbyo - fbya))/(so - s), fby = q6*q1 - q5*q2
            const double rh = nrcp(so - s);
            const double hy = ((so * o[6] - s * a[6]) - ((o[6] * o[1] - o[5] * o[2]) - (a[6] * a[1] - a[5] * a[2]))) * rh;
            const double hz = ((so * o[7] - s * a[7]) - ((o[7] * o[1] - o[5] * o[3]) - (a[7] * a[1] - a[5] * a[3]))) * rh;
            const double ny = hyb * rh, nz = hzb * rh;
            const double db = -((hyb * hy + hzb * hz) * rh);
            sob += (ny * o[6] + nz * o[7]) + db;
            sb -= (ny * a[6] + nz * a[7]) + db;
            ob[6] += ny * (so - o[1]);
            ob[7] += nz * (so - o[1]);
            ab[6] -= ny * (s - a[1]);
            ab[7] -= nz * (s - a[1]);
            ob[1] -= ny * o[6] + nz * o[7];
            ab[1] += ny * a[6] + nz * a[7];
            ob[5] += ny * o[2] + nz * o[3];
            ab[5] -= ny * a[2] + nz * a[3];
            ob[2] += ny * o[5];
            ab[2] -= ny * a[5];
            ob[3] += nz * o[5];
            ab[3] -= nz * a[5];
        }
        const double x = s - a[1], dn = a[0] * x, xo = so - o[1], dno = o[0] * xo;
        ab[5] += bbb * o[5];
        ob[5] += bbb * a[5];
        // prt = 0.5*((pta + dn*(sm - a1)) + (pto + dno*(sm - o1)))
        const double h = 0.5 * prtb;
        ptb += h;
        double ptob = h;
        dnb += h * (sm - a[1]);
        dnob += h * (sm - o[1]);
        smb += h * (dn + dno);
        ab[1] -= h * dn;
        ob[1] -= h * dno;
        smb -= ssmb + ssmob;
        sb += ssmb;
        sob += ssmob;
        // sm = ((dno*o1 - pto) - (dn*a1 - pta))/(dno - dn), or the mirror image of it
        if (degen) {
            sb += 0.5 * smb;
            sob += 0.5 * smb;
        } else {
            const double q = smb * nrcp(dno - dn);
            dnob += q * (o[1] - sm);
            dnb -= q * (a[1] - sm);
            ob[1] += q * dno;
            ab[1] -= q * dn;
            ptob -= q;
            ptb += q;
        }
        // dn = q0*x, x = s - q1
        ab[0] = (0.5 * enb) * ((a[1] * a[1] + a[2] * a[2]) + a[3] * a[3]) + dnb * x;
        xb += dnb * a[0];
        ob[0] = dnob * xo;
        xob += dnob * o[0];
        sb += xb;
        ab[1] -= xb;
        sob += xob;
        ob[1] -= xob;
        ab[4] = ptb + enb * rg1;
        ob[4] = ptob;
        double b2ab = 0.5 * (enb + ptb), b2ob = 0.5 * ptob;
        // sl = min(l1, r1) - c, sr = max(l1, r1) + c, c = sqrt(0.5*max(cl, cr))
        {
            const double lowb = left ? sb : sob, highb = left ? sob : sb;
            double wa, wo;
            dmin(a[1], o[1], wa, wo);
            ab[1] += lowb * wa;
            ob[1] += lowb * wo;
            dmax(a[1], o[1], wa, wo);
            ab[1] += highb * wa;
            ob[1] += highb * wo;
            // c_ = (t + sq)/q0 = 2*c*c on the larger side, sq = sqrt(t*t - 4*gp*q5^2), t = gp + b2, gp = gam*p
            const double cmb = (highb - lowb) * (((maxl && maxr) ? 0.125 : 0.25) * nrcp(cc));
            const double cm = 2.0 * (cc * cc);
            if (left ? maxl : maxr) {
                const double n = cmb * nrcp(a[0]);
                const double gp = gam * a[4], t = gp + ((a[5] * a[5] + a[6] * a[6]) + a[7] * a[7]);
                const double yb = n * (0.5 * nrcp(nsqrt(t * t - (4.0 * gp) * (a[5] * a[5]))));
                const double tb = n + (2.0 * yb) * t;
                ab[0] -= n * cm;
                ab[4] += (tb - (4.0 * yb) * (a[5] * a[5])) * gam;
                ab[5] -= (8.0 * yb) * (gp * a[5]);
                b2ab += tb;
            }
            if (left ? maxr : maxl) {
                const double n = cmb * nrcp(o[0]);
                const double gp = gam * o[4], t = gp + ((o[5] * o[5] + o[6] * o[6]) + o[7] * o[7]);
                const double yb = n * (0.5 * nrcp(nsqrt(t * t - (4.0 * gp) * (o[5] * o[5]))));
                const double tb = n + (2.0 * yb) * t;
                ob[0] -= n * cm;
                ob[4] += (tb - (4.0 * yb) * (o[5] * o[5])) * gam;
                ob[5] -= (8.0 * yb) * (gp * o[5]);
                b2ob += tb;
            }
        }
        b2ab *= 2.0;
        b2ob *= 2.0;
#pragma unroll
        for (int v = 5; v < 8; v++) {
            ab[v] += b2ab * a[v];
            ob[v] += b2ob * o[v];
        }
        if (!both || pass) break;
        // sm == 0: once more with the sides exchanged
        left = !left;
#pragma unroll
        for (int v = 0; v < 8; v++) {
            first[v] = ab[v];
            first[8 + v] = ob[v];
            swap_(a[v], o[v]);
        }
        swap_(s, so);
    }
    if (both) {
#pragma unroll
        for (int v = 0; v < 8; v++) {
            ab[v] += first[8 + v];
            ob[v] += first[v];
        }
    }
#pragma unroll
    for (int v = 0; v < 8; v++) {
        lb[v] += left ? ab[v] : ob[v];
        rb[v] += left ? ob[v] : ab[v];
    }
    return chb;
}

PK_HD double hlld_vjp(const double *l, const double *r, double gam, double ch, const double *fb, double *lb,
                      double *rb)
{
    return hlld_vjp_r(l, r, gam, 1.0 / gam, 1.0 / (gam - 1.0), ch, 1.0 / ch, fb, lb, rb);
}

// ---- utoq (MHD) ------------------------------------------------------------------
// q = prim<MHD>(u): HD part, then p -= (0.5*gam_1)*|B|^2, B and psi copied.
PK_HD void prim_vjp_mhd(const double (&u)[9], double gam_1, const double (&qb)[9], double (&ub)[9])
{
    const double a[5] = {u[0], u[1], u[2], u[3], u[4]};
    const double b[5] = {qb[0], qb[1], qb[2], qb[3], qb[4]};
    double o[5] = {0, 0, 0, 0, 0};
    prim_vjp_hd(a, gam_1, b, o);
#pragma unroll
    for (int v = 0; v < 5; v++) ub[v] += o[v];
    const double b2b = -((0.5 * gam_1) * qb[4]);
    ub[5] += qb[5] + 2.0 * u[5] * b2b;
    ub[6] += qb[6] + 2.0 * u[6] * b2b;
    ub[7] += qb[7] + 2.0 * u[7] * b2b;
    ub[8] += qb[8];
}

// floors<MHD>: as the HD floors with e = (E - kin) - mag, E = (e + kin) + mag.
PK_HD void floors_vjp_mhd(const double (&u)[9], double smalld, double smallei, int use_smalld, int use_smallei,
                          double (&ub)[9])
{
    double d = u[0];
    const bool dfl = use_smalld && !(d >= smalld);
    if (use_smalld) d = fmx(d, smalld);
    if (!use_smallei) {
        if (dfl) ub[0] = 0.0;
        return;
    }
    const double rd = nrcp(d);
    const double ek = ndiv(0.5 * ((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3]), d, rd);
    const double mag = 0.5 * ((u[5] * u[5] + u[6] * u[6]) + u[7] * u[7]);
    const double e = (u[4] - ek) - mag;
    const bool efl = !(e >= smallei);
    const double eb = efl ? 0.0 : ub[4];
    const double kb = ub[4] - eb;  // adjoint reaching kin and mag (they cancel when e is not floored)
    double db = ub[0];
    ub[4] = eb;
    const double sb = kb * rd;
    db -= sb * ek;
    ub[1] += sb * u[1];
    ub[2] += sb * u[2];
    ub[3] += sb * u[3];
    ub[5] += kb * u[5];
    ub[6] += kb * u[6];
    ub[7] += kb * u[7];
    ub[0] = dfl ? 0.0 : db;
}

// timestep_fluid at one cell, one direction (ion_cs, initionized.F90:137-141):
// t = dl / max(|m_q/rho| + cs, small), cs = sqrt(|(2 pmag + gam p)/rho|),
// p = ((E - ek)*(gam-1) + (2-gam)*pmag) - pmag.
PK_HD void dt_vjp_mhd(const double (&u)[9], int qdir, double dl, double gam, double gam_1, double tb,
                      double (&ub)[9])
{
    const double small = 1.17549435082228750797e-38;
    const double d = u[0];
    const double vq = (d > 0.0) ? fabs(u[1 + qdir] / d) : 0.0;
    const double ek = (0.5 * ((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3])) / d;
    const double pmag = 0.5 * ((u[5] * u[5] + u[6] * u[6]) + u[7] * u[7]);
    const double ps = (u[4] - ek) * gam_1 + (2.0 - gam) * pmag;
    const double pr = ps - pmag;
    const double x = (2.0 * pmag + gam * pr) / d;
    const double cs = sqrt(fabs(x));
    const double c = fmx(vq + cs, small);
    if (!(vq + cs > small)) return;
    const double cb = -(tb * dl) / (c * c);
    if (d > 0.0) {
        const double vv = u[1 + qdir] / d;
        const double sg = (vv > 0.0) ? 1.0 : ((vv < 0.0) ? -1.0 : 0.0);
        ub[1 + qdir] += cb * sg / d;
        ub[0] -= cb * sg * vv / d;
    }
    if (cs > 0.0) {
        const double sx = (x > 0.0) ? 1.0 : ((x < 0.0) ? -1.0 : 0.0);
        const double xb = cb * sx / (2.0 * cs);
        ub[0] -= xb * x / d;
        const double nb = xb / d;
        double pmb = 2.0 * nb;
        const double prb = nb * gam;
        // pr = ps - pmag; ps = (E - ek)*gam_1 + (2-gam)*pmag
        pmb += -prb + prb * (2.0 - gam);
        ub[4] += prb * gam_1;
        const double ekb = -(prb * gam_1);
        const double sb = ekb / d;
        ub[0] -= ekb * ek / d;
        ub[1] += sb * u[1];
        ub[2] += sb * u[2];
        ub[3] += sb * u[3];
        ub[5] += pmb * u[5];
        ub[6] += pmb * u[6];
        ub[7] += pmb * u[7];
    }
}

// ---- floors (HD) ---------------------------------------------------------------
// u_out = floors(u_in) (sources.F90:299-433): rho = max(rho, smalld); then
// e = E - ek, e = max(e, smallei), E = e + ek (always re-summed).
// Given ub = dL/du_out (in place), returns dL/du_in.
PK_HD void floors_vjp_hd(const double (&u)[5], double smalld, double smallei, int use_smalld, int use_smallei,
                         double (&ub)[5])
{
    double d = u[0];
    const bool dfl = use_smalld && !(d >= smalld);  // max(d, smalld) took smalld
    if (use_smalld) d = fmx(d, smalld);
    if (!use_smallei) {
        if (dfl) ub[0] = 0.0;
        return;
    }
    const double rd = nrcp(d);
    const double ek = ndiv(0.5 * ((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3]), d, rd);
    const double e = u[4] - ek;
    const bool efl = !(e >= smallei);
    // E_out = max(e, smallei) + ek
    const double eb = efl ? 0.0 : ub[4];
    const double ekb = ub[4] - eb;  // through "+ ek" and "e = E - ek"
    double db = ub[0];
    ub[4] = eb;
    const double sb = ekb * rd;
    db -= sb * ek;
    ub[1] += sb * u[1];
    ub[2] += sb * u[2];
    ub[3] += sb * u[3];
    ub[0] = dfl ? 0.0 : db;
}

// ---- timestep_fluid at one cell, one direction (HD, neu_cs) ----------------------
// t = dl / max(|m_q/rho| + cs, small), cs = sqrt(|gam*p/rho|),
// p = (E - ek)*(gam-1).  Given tb = dL/dt, add dL/du to ub.
PK_HD void dt_vjp_hd(const double (&u)[5], int qdir, double dl, double gam, double gam_1, double tb,
                     double (&ub)[5])
{
    const double small = 1.17549435082228750797e-38;
    const double d = u[0];
    const double vq = (d > 0.0) ? fabs(u[1 + qdir] / d) : 0.0;
    const double ek = (0.5 * ((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3])) / d;
    const double pr = (u[4] - ek) * gam_1;
    const double x = (gam * pr) / d;
    const double cs = sqrt(fabs(x));
    const double c = fmx(vq + cs, small);
    if (!(vq + cs > small)) return;
    const double cb = -(tb * dl) / (c * c);
    // vq = |m/d|
    if (d > 0.0) {
        const double vv = u[1 + qdir] / d;
        const double sg = (vv > 0.0) ? 1.0 : ((vv < 0.0) ? -1.0 : 0.0);
        ub[1 + qdir] += cb * sg / d;
        ub[0] -= cb * sg * vv / d;
    }
    // cs = sqrt(|x|)
    if (cs > 0.0) {
        const double sx = (x > 0.0) ? 1.0 : ((x < 0.0) ? -1.0 : 0.0);
        const double xb = cb * sx / (2.0 * cs);
        const double prb = xb * gam / d;
        ub[0] -= xb * x / d;
        ub[4] += prb * gam_1;
        const double ekb = -(prb * gam_1);
        const double sb = ekb / d;
        ub[0] -= ekb * ek / d;
        ub[1] += sb * u[1];
        ub[2] += sb * u[2];
        ub[3] += sb * u[3];
    }
}

}  // namespace PK_KNS
