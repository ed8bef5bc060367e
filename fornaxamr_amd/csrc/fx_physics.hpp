// Per-cell / per-face / per-edge physics of the RK2 Godunov stage, as device
// functions for gfx950.  FP64 throughout.
//
// Every expression keeps the operation order and association of the reference
// (cited per function) and the library is built with -ffp-contract=off, so the
// results are bit-identical to the reference CPU path whenever the FP64
// division and square root round correctly (they do on gfx950).  Min/max are
// written as the reference's ternaries, not fmin/fmax, to keep signed-zero and
// NaN behaviour identical.
#pragma once

#include <hip/hip_runtime.h>

#include "fx_log.hpp"

namespace fx {

// Largest of the workgroup's values (none of them NaN; blockDim.x a multiple
// of 64), returned to every thread.  lds: one double per wave of LDS that no
// thread touches until the next barrier after this call.
__device__ __forceinline__ double workgroup_max(double v, double* lds)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off);
        if (o > v) v = o;
    }
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = lds[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
        if (lds[w] > r) r = lds[w];
    return r;
}

__device__ __forceinline__ double dt_from_denom(double cfl, double max_denom)
{
    const double dt = cfl / max_denom;
    return dt < 1.0e99 ? dt : 1.0e99;
}

// dt = min(dt_new, factor * previous dt) after the first step (src/main.c:517-522)
__device__ __forceinline__ double growth_limit(double dt_new, double prev, double factor)
{
    if (prev > 0.0) {
        const double lim = factor * prev;
        return dt_new <= lim ? dt_new : lim;
    }
    return dt_new;
}

// The step's dt, by a whole workgroup, from the n recorded CFL maxima `part` and the
// previous dt; the same in every thread (a scalar).  lds as for workgroup_max.
__device__ __forceinline__ double form_step_dt(const double* part, int n, double cfl,
                                               double factor, double prev, double* lds)
{
    double best = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        if (part[i] > best) best = part[i];
    const double dt = growth_limit(dt_from_denom(cfl, workgroup_max(best, lds)), prev, factor);
    const long long b = __double_as_longlong(dt);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

// primitive / conserved variable slots (src/prj_defs.h:466-494)
enum { RHO = 0, V1 = 1, V2 = 2, V3 = 3, EINT = 4, YE = 5, B1 = 6, B2 = 7, B3 = 8 };
enum { MOM1 = 1, MOM2 = 2, MOM3 = 3, ETOT = 4 };

// local (face-frame) -> global primitive / conserved slot of direction dir
// (src/prj_flux.c:274-349): cyclic permutation of the vector components
__device__ __forceinline__ int gmap(int dir, int lv)
{
    if (lv == 0 || lv == 4 || lv == 5) return lv;
    if (lv <= 3) return 1 + (lv - 1 + dir) % 3;
    return 6 + (lv - 6 + dir) % 3;
}

__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }

// Half slope as the flux assembly uses it (src/prj_flux.c:410-418):
// h = 0.5 * prj_reconstruct_mc_face_slope(qm, q0, qp)
// (src/prj_reconstruct.h:355-375), evaluated as
//   (sl*sr > 0) ? 0.5 * copysign(min(|2 sl|, |c1|, |2 sr|), sl) : 0.
// When sl*sr > 0 the three candidates c0 = 2 sl, c1 = sl + (sr - sl)/2 and
// c2 = 2 sr are nonzero with the sign of sl, so min(c0,c1,c2) for sl > 0 and
// max(c0,c1,c2) for sl < 0 both equal copysign(min|c|, sl) exactly (negation
// and scaling by 2 are exact); otherwise both forms return +0.  Inputs with
// NaN give sl*sr > 0 false and 0 in both.  min(|2 sl|, |2 sr|) is taken as
// 2 min(|sl|, |sr|): doubling is exact (or overflows alike) and monotone, and
// a NaN c1 (from infinite slopes) is ignored by fmin in either order.  The
// same bits, half the instructions of the compare/select chain.
__device__ __forceinline__ double mc_half(double qm, double q0, double qp)
{
    double sl = q0 - qm;
    double sr = qp - q0;
    double c1 = sl + 0.5 * (sr - sl);
    double m = fmin(2.0 * fmin(fabs(sl), fabs(sr)), fabs(c1));
    double h = 0.5 * copysign(m, sl);
    return (sl * sr > 0.0) ? h : 0.0;
}

// The full MC face slope, prj_reconstruct_mc_face_slope (src/prj_reconstruct.h:
// 355-375), in the form of mc_half above: mc_half(...) == 0.5 * mc_slope(...)
// bit for bit (the same copysign(min|c|, sl), then the same product by 0.5).
__device__ __forceinline__ double mc_slope(double qm, double q0, double qp)
{
    double sl = q0 - qm;
    double sr = qp - q0;
    double c1 = sl + 0.5 * (sr - sl);
    double m = fmin(2.0 * fmin(fabs(sl), fabs(sr)), fabs(c1));
    double s = copysign(m, sl);
    return (sl * sr > 0.0) ? s : 0.0;
}

// Shock-detector pressure-jump limiter (src/prj_riemann.c:8-17).  The
// velocity deltas enter only through -min(., 0) + cfmax with cfmax > 0, so a
// min that differs from the reference's ternary only in the sign of a zero
// result gives the same theta; fmin (one instruction) is used throughout the
// delta chain.
__device__ __forceinline__ double theta_limiter(double cfmax, double du, double dv, double dw)
{
    double t = (-fmin(du, 0.0) + cfmax) / (-fmin(fmin(dv, dw), 0.0) + cfmax);
    t *= t;
    return fmin(1.0, t * t);
}

// min used for the velocity deltas (see theta_limiter)
__device__ __forceinline__ double dmin_delta(double a, double b) { return fmin(a, b); }

// The value of the next lane of this lane's row of 16: a DPP move, not a pass
// through LDS (ds_bpermute) that every wave would wait for right after the
// barrier (256^3 2.22 -> 2.20 ms per step, 96^3 160 -> 156 us).
__device__ __forceinline__ double next_in_row(double x)
{
    union { double d; int w[2]; } u = {x};
#pragma unroll
    for (int h = 0; h < 2; ++h) u.w[h] = __builtin_amdgcn_update_dpp(0, u.w[h], 0x101, 0xf, 0xf, true);
    return u.d;
}

// sqrt(a / b) with both operations correctly rounded, for a and b in
// [2^-300, 2^300] (sqrt_mid alone: [2^-601, 2^601]): Newton steps on the
// reciprocal and Markstein's correction of the quotient, then Goldschmidt's
// iteration on the square root with two such corrections (Markstein, IBM J. Res.
// Dev. 34, 1990).  The same steps as the full division and square root take once
// they have scaled their arguments, without the scaling and without the special
// cases: 18 instructions for 29
// (256^3 2.13 -> 2.11 ms per step, 128^3 HLLE 254 -> 246 us).
__device__ __forceinline__ double recip_mid(double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    return fma(fma(-b, r, 1.0), r, r);
}
// a / b, r = recip_mid(b)
__device__ __forceinline__ double quotient_mid(double a, double b, double r)
{
    const double x = a * r;
    return fma(fma(-b, x, a), r, x);
}
__device__ __forceinline__ double sqrt_mid(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double s = x * y, h = 0.5 * y;
    const double e = fma(-h, s, 0.5);
    s = fma(s, e, s);
    h = fma(h, e, h);
    s = fma(fma(-s, s, x), h, s);
    return fma(fma(-s, s, x), h, s);
}
__device__ __forceinline__ double sqrt_ratio_mid(double a, double b)
{
    return sqrt_mid(quotient_mid(a, b, recip_mid(b)));
}

// cL = sqrt(aL / rL), cR = sqrt(aR / rR).  Where all four numbers of every lane
// are well within the range (a NaN passes the test and comes out as one), the
// short form serves; else the full operations.  Same bits.
__device__ __forceinline__ void sound_speeds(double aL, double rL, double aR, double rR,
                                             double& cL, double& cR)
{
    const double lo = fmin(fmin(aL, rL), fmin(aR, rR)), hi = fmax(fmax(aL, rL), fmax(aR, rR));
    if (__builtin_amdgcn_ballot_w64(lo < 0x1p-300 || hi > 0x1p300) == 0) {
        cL = sqrt_ratio_mid(aL, rL);
        cR = sqrt_ratio_mid(aR, rR);
    } else {
        cL = sqrt(aL / rL);
        cR = sqrt(aR / rR);
    }
}

// HLLC with the theta-limited contact speed (src/prj_riemann.c:1433-1599),
// hydro build (6 variables).  W* are face states in the rotated frame.
//
// The reference returns F_L where 0 <= S_L, F_R
// where S_R <= 0, and otherwise the star flux of the side the contact speed
// selects (Toro 2009, eqs. 10.33-10.36).  Here the upwind side K is chosen
// once -- L if 0 <= S_L, R if S_R <= 0, else by the sign of S_M -- and F_K
// (formed from K's state by the same expressions as the reference's
// supersonic fluxes) is taken as it is in the supersonic cases and as the base
// of the star flux otherwise.  The star terms are added only where the
// reference would have formed them, so every returned bit is the reference's.
__device__ __forceinline__ void hllc(const double* WL, const double* WR, double pL, double pR,
                                     double gL, double gR, double du, double dv, double dw,
                                     double* flux, double* vface)
{
    // prj_riemann_state for both sides
    double rL = WL[RHO], uL = WL[V1], vL = WL[V2], wL = WL[V3], yL = WL[YE];
    double rR = WR[RHO], uR = WR[V1], vR = WR[V2], wR = WR[V3], yR = WR[YE];
    double eL = rL * WL[EINT] + 0.5 * rL * (uL * uL + vL * vL + wL * wL);
    double eR = rR * WR[EINT] + 0.5 * rR * (uR * uR + vR * vR + wR * wR);
    double csL, csR;
    sound_speeds(gL * pL, rL, gR * pR, rR, csL, csR);
    double UL1 = rL * uL, UR1 = rR * uR;

    double SL = dmin(uL - csL, uR - csR);
    double SR = dmax(uL + csL, uR + csR);
    double cfmax = dmax(csL, csR);
    double theta = theta_limiter(cfmax, du, dv, dw);
    double SM = (theta * (pR - pL) + UL1 * (SL - uL) - UR1 * (SR - uR)) /
                (rL * (SL - uL) - rR * (SR - uR));

    const bool sup_l = 0.0 <= SL;
    const bool sup_r = !sup_l && SR <= 0.0;
    const bool left = sup_l || (!sup_r && 0.0 <= SM);
    double r = left ? rL : rR;
    double u = left ? uL : uR;
    double v = left ? vL : vR;
    double w = left ? wL : wR;
    double y = left ? yL : yR;
    double e = left ? eL : eR;
    double p = left ? pL : pR;
    double S = left ? SL : SR;
    double Fr = r * u;
    double Fm1 = r * u * u + p;
    double Fm2 = r * u * v;
    double Fm3 = r * u * w;
    double Fe = (e + p) * u;
    double Fy = r * y * u;
    double rho_star = r * (S - u) / (S - SM);
    double e_over_rho = e / r + (SM - u) * (SM + p / (r * (S - u)));
    // The star terms are added under the lane mask: no select of 12 words per
    // face, and none of it where a wave is supersonic throughout (128^3 278 ->
    // 270 us per step, 112x48x80 91.8 -> 88.0).
    const double d0 = S * (rho_star - r);
    const double d1 = S * (rho_star * SM - r * u);
    const double d2 = S * (rho_star * v - r * v);
    const double d3 = S * (rho_star * w - r * w);
    const double d4 = S * (rho_star * e_over_rho - e);
    const double d5 = S * (rho_star * y - r * y);
    const bool sup = sup_l || sup_r;
    if (!sup) {
        Fr += d0;
        Fm1 += d1;
        Fm2 += d2;
        Fm3 += d3;
        Fe += d4;
        Fy += d5;
    }
    flux[0] = Fr;
    flux[1] = Fm1;
    flux[2] = Fm2;
    flux[3] = Fm3;
    flux[4] = Fe;
    flux[5] = Fy;
    vface[0] = sup ? u : SM;
    vface[1] = v;
    vface[2] = w;
}

// HLLE: the HLL flux (Harten, Lax & van Leer 1983) over the Davis wave-speed
// bounds SL = min(uL - cL, uR - cR), SR = max(uL + cL, uR + cR) that the
// reference's HLLC takes (src/prj_riemann.c:1518-1519), on the reference's
// face states (prj_riemann_state, src/prj_riemann.c:1433-1492).  The flux and
// the face velocity (that of the HLL average state) are written in the form of
// the reference's HLL fallback inside HLLD (src/prj_riemann.c:393-407).  Not
// a reference solver: the reference has no hydro HLLE.
__device__ __forceinline__ void hlle_hydro(const double* WL, const double* WR, double pL,
                                           double pR, double gL, double gR, double* flux,
                                           double* vface)
{
    double rL = WL[RHO], uL = WL[V1], vL = WL[V2], wL = WL[V3], yL = WL[YE];
    double rR = WR[RHO], uR = WR[V1], vR = WR[V2], wR = WR[V3], yR = WR[YE];
    double eL = rL * WL[EINT] + 0.5 * rL * (uL * uL + vL * vL + wL * wL);
    double eR = rR * WR[EINT] + 0.5 * rR * (uR * uR + vR * vR + wR * wR);
    double csL, csR;
    sound_speeds(gL * pL, rL, gR * pR, rR, csL, csR);
    double UL[6] = {rL, rL * uL, rL * vL, rL * wL, eL, rL * yL};
    double UR[6] = {rR, rR * uR, rR * vR, rR * wR, eR, rR * yR};
    double FL[6] = {rL * uL, rL * uL * uL + pL, rL * uL * vL, rL * uL * wL, (eL + pL) * uL,
                    rL * yL * uL};
    double FR[6] = {rR * uR, rR * uR * uR + pR, rR * uR * vR, rR * uR * wR, (eR + pR) * uR,
                    rR * yR * uR};
    double SL = dmin(uL - csL, uR - csR);
    double SR = dmax(uL + csL, uR + csR);
    // supersonic faces take the upwind flux in the place of the fan's, under the
    // lane mask (128^3 246 -> 240 us per step against selects)
    const bool sup_l = 0.0 <= SL;
    const bool sup_r = !sup_l && SR <= 0.0;
    const double inv = 1.0 / (SR - SL);
    double Uh[4];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        flux[v] = (SR * FL[v] - SL * FR[v] + SL * SR * (UR[v] - UL[v])) * inv;
        if (v < 4) Uh[v] = (SR * UR[v] - SL * UL[v] + FL[v] - FR[v]) * inv;
    }
    const double vh1 = Uh[1] / Uh[0], vh2 = Uh[2] / Uh[0], vh3 = Uh[3] / Uh[0];
    const bool sup = sup_l || sup_r;
    if (sup) {
#pragma unroll
        for (int v = 0; v < 6; ++v) flux[v] = sup_l ? FL[v] : FR[v];
    }
    vface[0] = sup ? (sup_l ? uL : uR) : vh1;
    vface[1] = sup ? (sup_l ? vL : vR) : vh2;
    vface[2] = sup ? (sup_l ? wL : wR) : vh3;
}

// ---- HLLD (src/prj_riemann.c:19-440) --------------------------------------

// Error codes mirror the reference abort sites.
enum HlldError {
    HLLD_OK = 0,
    HLLD_BAD_RHO = 11,       // src/prj_riemann.c:159-161
    HLLD_BAD_P = 12,         // :162-164
    HLLD_BAD_GAMMA = 13,     // :165-167
    HLLD_BAD_DISC = 14,      // :126-128
    HLLD_BAD_CF = 15,        // :131-133
    HLLD_BAD_ORDER = 16,     // :361-363
    HLLD_BAD_CONTACT = 17,   // :381-384
    HLLD_COINCIDE = 18,      // :198-200
    HLLD_BAD_STAR_RHO = 19,  // :203-205
    HLLD_BAD_DSS = 20        // :247-249
};

struct HlldSide {
    double rho, vx, vy, vz, by, bz, p, g, ye, e, pt;
};

struct HlldStar {
    double rho, vx, vy, vz, by, bz, ye, e;
};

// conserved vector of a state (src/prj_riemann.c:81-93)
__device__ __forceinline__ void hlld_cons(double rho, double vx, double vy, double vz, double bx,
                                          double by, double bz, double ye, double e, double* U)
{
    U[0] = rho;
    U[1] = rho * vx;
    U[2] = rho * vy;
    U[3] = rho * vz;
    U[4] = e;
    U[5] = rho * ye;
    U[6] = bx;
    U[7] = by;
    U[8] = bz;
}

// physical flux (src/prj_riemann.c:95-115)
__device__ __forceinline__ void hlld_flux(const HlldSide& s, double bx, double* F)
{
    const double pt = s.pt;   // p + 0.5 b^2, formed with the state
    double vdotb = s.vx * bx + s.vy * s.by + s.vz * s.bz;
    F[0] = s.rho * s.vx;
    F[1] = s.rho * s.vx * s.vx + pt - bx * bx;
    F[2] = s.rho * s.vx * s.vy - bx * s.by;
    F[3] = s.rho * s.vx * s.vz - bx * s.bz;
    F[4] = (s.e + pt) * s.vx - bx * vdotb;
    F[5] = s.rho * s.ye * s.vx;
    F[6] = 0.0;
    F[7] = s.by * s.vx - bx * s.vy;
    F[8] = s.bz * s.vx - bx * s.vz;
}

// state from primitives (src/prj_riemann.c:142-179)
__device__ __forceinline__ void hlld_side(const double* W, double p, double g, double bn,
                                          HlldSide& s)
{
    s.rho = W[RHO];
    s.vx = W[V1];
    s.vy = W[V2];
    s.vz = W[V3];
    s.by = W[B2];
    s.bz = W[B3];
    s.p = p;
    s.g = g;
    s.ye = W[YE];
    double kinetic = 0.5 * s.rho * (s.vx * s.vx + s.vy * s.vy + s.vz * s.vz);
    double magnetic = 0.5 * (bn * bn + s.by * s.by + s.bz * s.bz);
    s.e = s.rho * W[EINT] + kinetic + magnetic;
    s.pt = s.p + magnetic;
}

// the first failing check of a state (src/prj_riemann.c:159-167)
__device__ __forceinline__ int hlld_side_error(const HlldSide& s)
{
    if (s.rho <= 0.0) return HLLD_BAD_RHO;
    if (s.p <= 0.0) return HLLD_BAD_P;
    return s.g <= 0.0 ? HLLD_BAD_GAMMA : HLLD_OK;
}

// fast magnetosonic speed (src/prj_riemann.c:117-140); its checks go to bad_disc
// and bad_cf.  MID: rho and g p in [2^-300, 2^300], the squared fields there or zero:
// one reciprocal for the three quotients (of +0 the quotient is +0), and the short
// square root of cf2, which is at least half of a2.
template <bool MID>
__device__ __forceinline__ double hlld_fast(const HlldSide& s, double bx, bool& bad_disc,
                                            bool& bad_cf)
{
    const double r = MID ? recip_mid(s.rho) : 0.0;
    const auto over_rho = [&](double a) { return MID ? quotient_mid(a, s.rho, r) : a / s.rho; };
    double a2 = over_rho(s.g * s.p);
    double bx2_rho = over_rho(bx * bx);
    double b2_rho = over_rho(bx * bx + s.by * s.by + s.bz * s.bz);
    double disc = (a2 + b2_rho) * (a2 + b2_rho) - 4.0 * a2 * bx2_rho;
    bad_disc = disc < 0.0 && disc < -1.0e-12 * (a2 + b2_rho) * (a2 + b2_rho);
    disc = disc < 0.0 ? 0.0 : disc;
    double cf2 = 0.5 * (a2 + b2_rho + sqrt(disc));
    bad_cf = cf2 < 0.0 || !isfinite(cf2);
    return MID ? sqrt_mid(cf2) : sqrt(cf2);
}

// whether every lane's pair of states is in the range of hlld_fast<true>
__device__ __forceinline__ bool hlld_mid(const HlldSide& L, const HlldSide& R, double bx)
{
    const double gpL = L.g * L.p, gpR = R.g * R.p;
    const double lo = fmin(fmin(gpL, L.rho), fmin(gpR, R.rho));
    const double b0 = bx * bx, bL = b0 + L.by * L.by + L.bz * L.bz,
                 bR = b0 + R.by * R.by + R.bz * R.bz;
    const double hi = fmax(fmax(fmax(gpL, L.rho), fmax(gpR, R.rho)), fmax(bL, bR));
    unsigned long long out = __builtin_amdgcn_ballot_w64(lo < 0x1p-300 || hi > 0x1p300);
    for (const double b : {b0, bL, bR})
        out |= __builtin_amdgcn_ballot_w64(b < 0x1p-300) & ~__builtin_amdgcn_ballot_w64(b == 0.0);
    return out == 0;
}

// outer (single-star) state (src/prj_riemann.c:187-232)
__device__ __forceinline__ int hlld_outer(const HlldSide& s, double bx, double S, double SM,
                                          double pt_star, HlldStar& st)
{
    double alpha = S - s.vx;
    double smdiff = S - SM;
    const bool coincide = fabs(smdiff) <= 1.0e-14 * (fabs(S) + fabs(SM) + 1.0);
    st.rho = s.rho * alpha / smdiff;
    const bool bad = coincide | (st.rho <= 0.0) | !isfinite(st.rho);
    st.vx = SM;
    st.ye = s.ye;
    double denom = s.rho * alpha * smdiff - bx * bx;
    if (fabs(denom) < 1.0e-8 * pt_star) {
        st.vy = s.vy;
        st.vz = s.vz;
        st.by = s.by;
        st.bz = s.bz;
    } else {
        double q = (SM - s.vx) / denom;
        double mag = (s.rho * alpha * alpha - bx * bx) / denom;
        st.vy = s.vy - bx * s.by * q;
        st.vz = s.vz - bx * s.bz * q;
        st.by = s.by * mag;
        st.bz = s.bz * mag;
    }
    double vdotb = s.vx * bx + s.vy * s.by + s.vz * s.bz;
    double vsdotbs = st.vx * bx + st.vy * st.by + st.vz * st.bz;
    st.e = (alpha * s.e - s.pt * s.vx + pt_star * SM + bx * (vdotb - vsdotbs)) / smdiff;
    return bad ? (coincide ? HLLD_COINCIDE : HLLD_BAD_STAR_RHO) : HLLD_OK;
}

// HLLD flux (src/prj_riemann.c:321-440).  WL/WR are rotated face states with
// the normal field slot already set to bn.  Outputs the 9-variable flux, the
// face velocity and the face EMFs Bv1 = bz*vx - bx*vz, Bv2 = bx*vy - by*vx of
// the selected fan state (src/prj_riemann.c:305-319).  On an error the outputs
// mean nothing, but every one of them is set.
//
// Bound by instruction issue: a return behind each of the reference's dozen
// checks cut the solver into as many masked regions, between which nothing is
// scheduled.  One branch holds the checks of both states, and the supersonic, single-
// and double-star fluxes are stages of one sum rather than separate exits.
// MHD step: 256^3 7.54 -> 6.87 ms, 128^3 1041 -> 957 us, 48x32x64 120 -> 114.
// SHORT: with the short forms of the fast speeds (256^3 7.00 -> 6.88 ms per step on a
// slower card, 112x48x80 274 -> 268 us; not worth it in the per-block kernel, whose one
// workgroup per CU of 8 waves gains nothing: 343 blocks 390 -> 392 us).
template <bool SHORT = true>
__device__ __forceinline__ int hlld(const double* WL, const double* WR, double pL, double pR,
                                 double gL, double gR, double bn, double* flux, double* vface,
                                 double* bv1, double* bv2)
{
    HlldSide L, R;
    int rc;
    const auto refused = [&](int code) {
        for (int v = 0; v < 9; ++v) flux[v] = 0.0;
        vface[0] = vface[1] = vface[2] = *bv1 = *bv2 = 0.0;
        return code;
    };
    hlld_side(WL, pL, gL, bn, L);
    hlld_side(WR, pR, gR, bn, R);
    bool bad[4];
    double cfL, cfR;
    if (SHORT && hlld_mid(L, R, bn)) {
        cfL = hlld_fast<true>(L, bn, bad[0], bad[1]);
        cfR = hlld_fast<true>(R, bn, bad[2], bad[3]);
    } else {
        cfL = hlld_fast<false>(L, bn, bad[0], bad[1]);
        cfR = hlld_fast<false>(R, bn, bad[2], bad[3]);
    }
    double SL = dmin(L.vx - cfL, R.vx - cfR);
    double SR = dmax(L.vx + cfL, R.vx + cfR);
    // one branch for the checks of both states: what follows a failed one is
    // garbage, and the first of them in the reference's order is the result
    const bool any = (L.rho <= 0.0) | (L.p <= 0.0) | (L.g <= 0.0) | (R.rho <= 0.0) |
                     (R.p <= 0.0) | (R.g <= 0.0) | bad[0] | bad[1] | bad[2] | bad[3] |
                     !(SL < SR);
    if (any) {
        rc = HLLD_BAD_ORDER;
        for (int c = 3; c >= 0; --c)
            if (bad[c]) rc = c & 1 ? HLLD_BAD_CF : HLLD_BAD_DISC;
        if (const int e = hlld_side_error(R)) rc = e;
        if (const int e = hlld_side_error(L)) rc = e;
        return refused(rc);
    }

    const bool sup_l = 0.0 <= SL;
    const bool sup = sup_l || SR <= 0.0;
    double denom = R.rho * (SR - R.vx) - L.rho * (SL - L.vx);
    if (!sup && fabs(denom) <= 1.0e-14 * (fabs(R.rho * (SR - R.vx)) +
                                          fabs(L.rho * (SL - L.vx)) + 1.0))
        return refused(HLLD_BAD_CONTACT);
    double SM = (R.rho * R.vx * (SR - R.vx) - L.rho * L.vx * (SL - L.vx) + (L.pt - R.pt)) / denom;
    double ptl = L.pt + L.rho * (SL - L.vx) * (SM - L.vx);
    double ptr = R.pt + R.rho * (SR - R.vx) * (SM - R.vx);
    double pt_star = 0.5 * (ptl + ptr);
    if (!sup && (pt_star <= 0.0 || !isfinite(pt_star))) {
        // HLL fallback (src/prj_riemann.c:393-407): both outer states needed
        double UL[9], UR[9], FL[9], FR[9];
        hlld_flux(L, bn, FL);
        hlld_flux(R, bn, FR);
        hlld_cons(L.rho, L.vx, L.vy, L.vz, bn, L.by, L.bz, L.ye, L.e, UL);
        hlld_cons(R.rho, R.vx, R.vy, R.vz, bn, R.by, R.bz, R.ye, R.e, UR);
        double inv = 1.0 / (SR - SL);
        double Uh[9];
        for (int v = 0; v < 9; ++v) {
            flux[v] = (SR * FL[v] - SL * FR[v] + SL * SR * (UR[v] - UL[v])) * inv;
            Uh[v] = (SR * UR[v] - SL * UL[v] + FL[v] - FR[v]) * inv;
        }
        double rho = Uh[0];
        double vx = Uh[1] / rho, vy = Uh[2] / rho, vz = Uh[3] / rho;
        vface[0] = vx; vface[1] = vy; vface[2] = vz;
        *bv1 = Uh[8] * vx - Uh[6] * vz;
        *bv2 = Uh[6] * vy - Uh[7] * vx;
        return HLLD_OK;
    }
    // The upwind outer side A: the upstream one of a supersonic face, else the
    // contact's.  Its flux and state are what the star terms below, added under
    // the lane mask, start from.
    const bool left = sup ? sup_l : 0.0 <= SM;
    const HlldSide& A = left ? L : R;
    double FA[9];
    hlld_flux(A, bn, FA);
    double vx = A.vx, vy = A.vy, vz = A.vz, by = A.by, bz = A.bz;
    rc = HLLD_OK;
    if (!sup) {
        const double SA = left ? SL : SR;
        double UA[9];
        hlld_cons(A.rho, A.vx, A.vy, A.vz, bn, A.by, A.bz, A.ye, A.e, UA);
        HlldStar As;
        rc = hlld_outer(A, bn, SA, SM, pt_star, As);
        double sqA = sqrt(As.rho);
        double SAs = left ? SM - fabs(bn) / sqA : SM + fabs(bn) / sqA;
        double UAs[9];
        hlld_cons(As.rho, As.vx, As.vy, As.vz, bn, As.by, As.bz, As.ye, As.e, UAs);
        for (int v = 0; v < 9; ++v) FA[v] = FA[v] + SA * (UAs[v] - UA[v]);
        vx = As.vx; vy = As.vy; vz = As.vz; by = As.by; bz = As.bz;
        // The other side's star state is only needed for the double-star
        // (rotational) state (src/prj_riemann.c:234-282).
        const bool bn_small = (0.5 * bn * bn < 1.0e-8 * pt_star);
        if (rc == HLLD_OK && !(left ? 0.0 <= SAs : SAs <= 0.0) && !bn_small) {
            const HlldSide& Bo = left ? R : L;
            const double SB = left ? SR : SL;
            HlldStar Bs;
            rc = hlld_outer(Bo, bn, SB, SM, pt_star, Bs);
            const HlldStar& Ls = left ? As : Bs;
            const HlldStar& Rs = left ? Bs : As;
            const double sqB = sqrt(Bs.rho);
            const double sl = left ? sqA : sqB;
            const double sr = left ? sqB : sqA;
            if (rc == HLLD_OK && sl + sr <= 0.0) rc = HLLD_BAD_DSS;
            double inv_sum = 1.0 / (sl + sr);
            double sgn = bn < 0.0 ? -1.0 : 1.0;
            vy = (sl * Ls.vy + sr * Rs.vy + (Rs.by - Ls.by) * sgn) * inv_sum;
            vz = (sl * Ls.vz + sr * Rs.vz + (Rs.bz - Ls.bz) * sgn) * inv_sum;
            by = (sl * Rs.by + sr * Ls.by + sl * sr * (Rs.vy - Ls.vy) * sgn) * inv_sum;
            bz = (sl * Rs.bz + sr * Ls.bz + sl * sr * (Rs.vz - Ls.vz) * sgn) * inv_sum;
            double vbss = As.vx * bn + vy * by + vz * bz;
            const double vba = As.vx * bn + As.vy * As.by + As.vz * As.bz;
            const double ess = left ? As.e - sqA * sgn * (vba - vbss)
                                    : As.e + sqA * sgn * (vba - vbss);
            double Uss[9];
            hlld_cons(As.rho, As.vx, vy, vz, bn, by, bz, As.ye, ess, Uss);
            for (int v = 0; v < 9; ++v) FA[v] = FA[v] + SAs * (Uss[v] - UAs[v]);
        }
    }
    for (int v = 0; v < 9; ++v) flux[v] = FA[v];
    vface[0] = vx; vface[1] = vy; vface[2] = vz;
    *bv1 = bz * vx - bn * vz;
    *bv2 = bn * vy - by * vx;
    return rc;
}

// What the CT step needs of a double in 32 bits: its sign, whether it is zero and
// whether it is finite.  The high word, with its lowest bit set where the low word
// is not zero, so that no nonzero value looks like zero.
struct SignWord {
    int w;
};
__device__ __forceinline__ SignWord sign_word(double v)
{
    const long long b = __double_as_longlong(v);
    return {(int)(b >> 32) | ((int)b != 0 ? 1 : 0)};
}
__device__ __forceinline__ bool is_positive(double v) { return v > 0.0; }
__device__ __forceinline__ bool is_negative(double v) { return v < 0.0; }
// (of finite values; a word that is not finite is reported before its sign matters)
__device__ __forceinline__ bool is_positive(SignWord v) { return v.w > 0; }
__device__ __forceinline__ bool is_negative(SignWord v) { return (unsigned)v.w > 0x80000000u; }
__device__ __forceinline__ bool is_finite(SignWord v) { return (v.w & 0x7ff00000) != 0x7ff00000; }

// Upwind CT edge EMF without the resistive term (src/prj_mhd.c:651-683).
// The normal velocities enter by their signs only: V is double, or SignWord.
template <typename V>
__device__ __forceinline__ double emf_upwind(const double* ef, const double* ec, const V* vn)
{
    double emf = 0.25 * (ef[0] + ef[1] + ef[2] + ef[3]);
    if (is_positive(vn[0]))      emf += 0.25 * (ef[3] - ec[3]);
    else if (is_negative(vn[0])) emf += 0.25 * (ef[1] - ec[0]);
    else                  emf += 0.125 * (ef[3] - ec[3] + ef[1] - ec[0]);
    if (is_positive(vn[1]))      emf += 0.25 * (ef[2] - ec[1]);
    else if (is_negative(vn[1])) emf += 0.25 * (ef[0] - ec[0]);
    else                  emf += 0.125 * (ef[2] - ec[1] + ef[0] - ec[0]);
    if (is_positive(vn[2]))      emf += 0.25 * (ef[3] - ec[2]);
    else if (is_negative(vn[2])) emf += 0.25 * (ef[1] - ec[1]);
    else                  emf += 0.125 * (ef[3] - ec[2] + ef[1] - ec[1]);
    if (is_positive(vn[3]))      emf += 0.25 * (ef[2] - ec[2]);
    else if (is_negative(vn[3])) emf += 0.25 * (ef[0] - ec[3]);
    else                  emf += 0.125 * (ef[2] - ec[2] + ef[0] - ec[3]);
    return emf;
}

// Anomalous resistivity mask of one cell (src/prj_timeint.c:230-263):
// 1e12 * max(0, log(rho / 1e13)) * max(0, log(Ye / 0.25)).  A log factor is
// positive only when its argument exceeds 1 and is then taken with the
// correctly rounded log_cr (fx_log.hpp); at or below 1 every faithful log is
// <= 0 and the factor is 0, so the log is skipped there.  The reference aborts
// on a non-finite mask; none arises: each factor is at most
// log(DBL_MAX) < 710, so the mask stays below 1e12 * 710^2.  The quotients
// are formed only past the thresholds: rounding is monotone, so rho <= 1e13
// gives rho / 1e13 <= 1 (and ye / 0.25 is exact), and the factors are 0
// there without a division.  A factor of 0 makes the mask 0 (the other is finite),
// so the logs are taken only where both are positive, by one copy of the code.
__device__ __forceinline__ double eta_mask(double rho, double ye)
{
    if (!(rho > 1.0e13 && isfinite(rho) && ye > 0.25 && isfinite(ye))) return 0.0;
    const double x[2] = {rho / 1.0e13, ye / 0.25};
    double f[2] = {0.0, 0.0};
#pragma unroll 1
    for (int n = 0; n < 2; ++n)
        if ((n == 0 ? x[0] : x[1]) > 1.0) (n == 0 ? f[0] : f[1]) = log_cr(n == 0 ? x[0] : x[1]);
    return 1.0e12 * f[0] * f[1];
}

}  // namespace fx
