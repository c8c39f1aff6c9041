// Reverse mode of hllcFace() (icsf_flux.h; hllcFluxScheme.C:70-240) without a
// frame velocity, for the residual adjoint: one forward evaluation of the
// wave speeds, then one backward sweep.
//
// The flux is cSl F_L + cSlm F*_L + cSmr F*_R + cSr F_R with weights of 0 or
// 1.  cSlm needs Sm > 0 and cSmr Sm <= 0, so at most one star state counts:
// its side is selected first and its reverse written once (lanes of a
// wavefront on either side of a contact take the same instructions).
// Branches (min/max of the wave speeds, |x|, the VSMALL clips) follow the
// value the forward takes; ties take the first argument.
#pragma once
#include "icsf_math.h"
#include "icsf_views.h"

namespace icsf {

#define DFR __device__ __forceinline__

// L, R: owner- and neighbour-side face values [NFLD] (F_CS: the sound
// speed); (bphi, bphiU, bphiE): adjoint of the face flux; out: adjoints of
// the face values (bL, bR) and of Sf (bS, |Sf| taken as |Sf|(Sf)); branches
// (optional): bit 0 Sl = ua - ca, 1 Sr = ua + ca, 2 Sl > 0, 3 Sr < 0, 4
// Sm > 0, 5 the argument of ca's square root below zero.
DFR void hllcFaceRev(double gI, V3 S, const double* L, const double* R, double bphi, V3 bphiU, double bphiE,
                     double* bL, double* bR, V3& bS, int* branches) {
    const double rl = L[F_RHO], rr = R[F_RHO], pl = L[F_P], pr = R[F_P], cl = L[F_CS], cr = R[F_CS];
    const double El = L[F_E], Er = R[F_E], Hl = L[F_H], Hr = R[F_H];
    const V3 Ul{L[F_UX], L[F_UY], L[F_UZ]}, Ur{R[F_UX], R[F_UY], R[F_UZ]};

    // ---- forward: wave speeds
    const double magS = mag(S);
    const V3 n = S / magS;
    const bool freeR = kVSMALL < rr, freeL = kVSMALL < rl;
    const double al = freeL ? rl : kVSMALL, q = (freeR ? rr : kVSMALL) / al;
    const double k = sqrt(q), k1 = k + 1.0;
    const V3 uAvg = (k * Ur + Ul) / k1;
    const double HAvg = (k * Hr + Hl) / k1;
    const double arg = (gI - 1.0) * (HAvg - 0.5 * magSqr(uAvg));
    const double ca = sqrt(fabs(arg));
    const double ul = dot(Ul, n), ur = dot(Ur, n), ua = dot(uAvg, n);
    const bool slA = ua - ca < ul - cl, srA = ur + cr < ua + ca;
    const double Sl = slA ? ua - ca : ul - cl, Sr = srA ? ua + ca : ur + cr;
    const double den = rr * (Sr - ur) - rl * (Sl - ul);
    const double Sm = (rr * ur * (Sr - ur) - rl * ul * (Sl - ul) + pl - pr) / den;
    const bool left = Sm > 0;  // the side of the star state
    const bool outL = Sl > 0, outR = Sr < 0;
    if (branches)
        *branches = (int)slA | (int)srA << 1 | (int)outL << 2 | (int)outR << 3 | (int)left << 4 | (int)(arg < 0) << 5;

    // ---- reverse, (gm, gu, ge): adjoint of the flux per unit area
    const double gm = bphi * magS, ge = bphiE * magS;
    const V3 gu = bphiU * magS;
    V3 nB{0, 0, 0}, UlB{0, 0, 0}, UrB{0, 0, 0};
    double rlB = 0, rrB = 0, plB = 0, prB = 0, ulB = 0, urB = 0, HlB = 0, HrB = 0, ElB = 0, ErB = 0;
    double SmB = 0, SlB = 0, SrB = 0, magB = 0;
    // a side's own flux (rho u, rho u U + p n, rho H u)
    auto side = [&](double r, double p, V3 U, double u, double H, double& rB, double& pB, V3& UB, double& uB,
                    double& HB) {
        const double gU = dot(gu, U), t = gm + gU + ge * H;
        rB += u * t;
        uB += r * t;
        UB = UB + (r * u) * gu;
        pB += dot(gu, n);
        nB = nB + p * gu;
        HB += ge * r * u;
        magB += bphi * (r * u) + r * u * dot(bphiU, U) + p * dot(bphiU, n) + bphiE * (r * H * u);
    };
    if (outL) side(rl, pl, Ul, ul, Hl, rlB, plB, UlB, ulB, HlB);
    if (outR) side(rr, pr, Ur, ur, Hr, rrB, prB, UrB, urB, HrB);
    if (left ? !outL : !outR) {
        // the star state: qs = (Ss - us) r, inv = 1 / (Ss - Sm),
        //   mass Sm inv qs; ps = r (us - Ss) (us - Sm) + p,
        //   m = inv (qs U + (ps - p) n), momentum Sm m + ps n;
        //   e = inv (qs E - p us + ps Sm), energy Sm (e + ps)
        const double Ss = left ? Sl : Sr, us = left ? ul : ur, r = left ? rl : rr, p = left ? pl : pr;
        const double E = left ? El : Er;
        const V3 U = left ? Ul : Ur;
        const double inv = 1.0 / (Ss - Sm), qs = (Ss - us) * r;
        const double ps = r * (us - Ss) * (us - Sm) + p;
        const V3 mv = qs * U + (ps - p) * n;
        const V3 m = inv * mv;
        const double ev = qs * E - p * us + ps * Sm;
        const double e = inv * ev;
        magB += bphi * (Sm * inv * qs) + dot(bphiU, Sm * m + ps * n) + bphiE * (Sm * (e + ps));
        const double gn = dot(gu, n), gU = dot(gu, U);
        const double eB = ge * Sm;
        SmB += gm * inv * qs + dot(gu, m) + ge * (e + ps) + eB * inv * ps;
        const double invB = gm * Sm * qs + Sm * dot(gu, mv) + eB * ev;
        const double qsB = gm * Sm * inv + Sm * inv * gU + eB * inv * E;
        const double psB = gn + Sm * inv * gn + ge * Sm + eB * inv * Sm;
        const V3 UB = (Sm * inv * qs) * gu;
        nB = nB + (ps + Sm * inv * (ps - p)) * gu;
        const double EB = eB * inv * qs;
        const double dI = invB * inv * inv;
        SmB += dI - psB * r * (us - Ss);
        const double SsB = -dI - psB * r * (us - Sm) + qsB * r;
        const double usB = -eB * inv * p + psB * r * ((us - Sm) + (us - Ss)) - qsB * r;
        const double rB = psB * (us - Ss) * (us - Sm) + qsB * (Ss - us);
        const double pB = psB - Sm * inv * gn - eB * inv * us;
        if (left) { SlB += SsB; ulB += usB; rlB += rB; plB += pB; UlB = UlB + UB; ElB += EB; }
        else { SrB += SsB; urB += usB; rrB += rB; prB += pB; UrB = UrB + UB; ErB += EB; }
        // Sm = num / den
        const double numB = SmB / den, denB = -numB * Sm;
        rrB += numB * ur * (Sr - ur) + denB * (Sr - ur);
        urB += numB * rr * (Sr - 2.0 * ur) - denB * rr;
        SrB += numB * rr * ur + denB * rr;
        rlB -= numB * ul * (Sl - ul) + denB * (Sl - ul);
        ulB += denB * rl - numB * rl * (Sl - 2.0 * ul);
        SlB -= numB * rl * ul + denB * rl;
        plB += numB;
        prB -= numB;
    }
    // wave speeds
    double uaB = 0, caB = 0, clB = 0, crB = 0;
    if (slA) { uaB += SlB; caB -= SlB; }
    else { ulB += SlB; clB -= SlB; }
    if (srA) { uaB += SrB; caB += SrB; }
    else { urB += SrB; crB += SrB; }
    double argB = ca > 0.0 ? caB / (2.0 * ca) : 0.0;
    if (arg < 0.0) argB = -argB;
    const double HaB = (gI - 1.0) * argB;
    const V3 uaV = uaB * n - HaB * uAvg;
    nB = nB + uaB * uAvg + ulB * Ul + urB * Ur;
    UlB = UlB + ulB * n + uaV / k1;
    UrB = UrB + urB * n + (k / k1) * uaV;
    HlB += HaB / k1;
    HrB += HaB * k / k1;
    const double kB = (dot(uaV, Ur - uAvg) + HaB * (Hr - HAvg)) / k1;
    const double qB = k > 0.0 ? kB / (2.0 * k) : 0.0;
    if (freeR) rrB += qB / al;
    if (freeL) rlB -= qB * q / al;
    bS = nB / magS + (magB - dot(nB, n) / magS) * n;
    bL[F_RHO] = rlB; bL[F_P] = plB; bL[F_UX] = UlB.x; bL[F_UY] = UlB.y; bL[F_UZ] = UlB.z;
    bL[F_E] = ElB; bL[F_H] = HlB; bL[F_CS] = clB;
    bR[F_RHO] = rrB; bR[F_P] = prB; bR[F_UX] = UrB.x; bR[F_UY] = UrB.y; bR[F_UZ] = UrB.z;
    bR[F_E] = ErB; bR[F_H] = HrB; bR[F_CS] = crB;
}

#undef DFR
}  // namespace icsf
