// Differentiable hydro scheme and its hand-written discrete adjoint.
//
// Scheme (not in the reference, which has MC/WENO and HLLC/HLLD): PLM with the
// smooth van Albada slope  (sl (sr^2+e) + sr (sl^2+e)) / (sl^2+sr^2+2e),
// reconstructing rho, v, p = (gamma-1) rho eint and Ye; HLLE fluxes with the
// Davis speeds of src/prj_riemann.c:1518-1519 in the HLL form of
// src/prj_riemann.c:393-407; flux divergence and per-cell RK2 update as in
// src/prj_flux.c:2523-2533 and src/prj_timeint.c:1255-1350, 1562-1655; fixed
// dt; periodic box.  The forward kernels round exactly as the CPU oracle of
// the same scheme.
//
// Work split.  Along z, lanes hold consecutive cells of the rows and take their
// neighbours' face states from the lanes beside them; windows of 64 lanes overlap
// by the lanes that lack neighbours.  Along x and y windows of 32 positions x 8
// cells exchange through LDS.  So every slope and face is formed once, but for the
// overlaps.  A stage is two launches: the x and y directions, then the z direction
// and the sum at each cell.  Bound: half by the FP64 instructions, half by the
// 113 MB (forward) and 155 MB (reverse) that a 64^3 stage moves, at 5 TB/s.
// us at 64^3: forward stage 15.4 + 12.5, reverse stage 28.1 + 21.5; a face kernel
// and a cell kernel, all face values or cotangents through memory and each slope
// formed by every face that uses it, took 22 + 11 and 33 + 43.  One forward launch
// in which a lane formed both its x- and y-faces took 34 (2711 instructions a
// cell), threads marching 8-cell segments along x and y 21.5 + 10.6.
//
// Layout: compact cell fields [var][X][Y][Z] (Z fastest), var = rho, v1, v2,
// v3, eint, Ye; N = X*Y*Z.  Periodic neighbours by index wrap, no ghosts.
//
// Adjoint.  A stage maps  Wout = prim(a cons(Wa) + b (cons(Wb) + dt L(Wb))).
// The cotangent is carried in conserved variables, Ubar = Jprim(W)^T Wbar;
// then for RK2 (stage 1: a = 0, b = 1 from W0; stage 2: a = b = 1/2 from W0,
// W1), with dL(W)^T taken through the per-face HLLE and per-cell slope VJPs:
//   Ubar1 = 1/2 Ubar2 + Jprim(W1)^T dL(W1)^T (dt/2 Ubar2)
//   Ubar0 = 1/2 Ubar2 + Ubar1 + Jprim(W0)^T dL(W0)^T (dt Ubar1)
// (Jprim(W)^T Jcons(W)^T = I removes the cons() terms).  At an exact tie of a
// min/max the cotangent is split evenly between both operands.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fx_kernels.hpp"

namespace fx {
namespace {

constexpr int NT = 256;

// Quotients by one divisor: its reciprocal by two Newton-Raphson steps from the
// hardware's estimate, and per quotient the residual correction of Markstein
// (IBM J. Res. Dev. 34, 1990).  The divisor is scaled into [1, 2) first, so that
// nothing over- or underflows on the way that does not in the quotient; the fixup
// gives zeros, infinities and NaN as the division does.  7 + 5 instructions per
// quotient for 11 per division (40 steps and their reverse at 64^3 8.41 ms, by
// divisions 8.75; unguarded 8.33).
//
// The quotients are those of the division, to the bit, where every numerator is 0
// or at least 2^-961 (its residual is then a number) and every quotient is normal.
// exact() is whether that holds for all quotients formed so far in all lanes of
// the wave; where it does not, the forward kernels form them again by division
// (SHORT false), so that they round exactly whatever the state.  The reverse
// kernels, which round as they like (hlle_vjp multiplies by a reciprocal), do not
// ask: a quotient below that is off by a few units of the last place, or of the
// smallest subnormal where the numerator is one.
template <bool SHORT = true>
struct Recip {
    double b, m, y;
    int e;
    int least = 0;           // smallest exponent of a numerator (frexp's)
    __device__ __forceinline__ explicit Recip(double x) : b(x)
    {
        if (!SHORT) return;
        e = 1 - __builtin_amdgcn_frexp_exp(x);
        m = ldexp(x, e);
        y = __builtin_amdgcn_rcp(m);
        y = fma(y, fma(-m, y, 1.0), y);
        y = fma(y, fma(-m, y, 1.0), y);
    }
    __device__ __forceinline__ double operator()(double a)
    {
        if (!SHORT) return a / b;
        least = min(least, __builtin_amdgcn_frexp_exp(a));
        double q = a * y;
        q = fma(fma(-m, q, a), y, q);
        return __builtin_amdgcn_div_fixup(ldexp(q, e), b, a);
    }
    __device__ __forceinline__ bool exact() const
    {
        return !SHORT || __builtin_amdgcn_ballot_w64(least < max(-960, -1019 - e)) == 0;
    }
};

__device__ __forceinline__ int wrap(int i, int n)
{
    return i < 0 ? i + n : (i >= n ? i - n : i);
}

__device__ __forceinline__ double va(double sl, double sr, double e)
{
    const double sl2 = sl * sl, sr2 = sr * sr;
    const double num = sl * (sr2 + e) + sr * (sl2 + e);
    const double den = (sl2 + sr2) + 2.0 * e;
    return num / den;
}

// value and partial derivatives of the van Albada slope
__device__ __forceinline__ double va_d(double sl, double sr, double e, double& dl, double& dr)
{
    const double sl2 = sl * sl, sr2 = sr * sr;
    const double num = sl * (sr2 + e) + sr * (sl2 + e);
    Recip<> den((sl2 + sr2) + 2.0 * e);
    const double v = den(num);
    const double two_lr = 2.0 * sl * sr;
    dl = den((sr2 + e) + two_lr - v * (2.0 * sl));
    dr = den(two_lr + (sl2 + e) - v * (2.0 * sr));
    return v;
}

// rotated variable r of direction d: rho, v_n, v_t1, v_t2, p, Ye
__device__ __forceinline__ int rmap(int d, int r)
{
    if (r == 0) return 0;
    if (r >= 4) return r;
    return 1 + (d + r - 1) % 3;
}

struct HlleState {
    double U[6], F[6];
};

template <typename Q>
__device__ __forceinline__ void hlle_side(const double* a, Q& gm1, HlleState& s)
{
    const double m = a[0] * a[1];
    const double ke = (0.5 * a[0]) * ((a[1] * a[1] + a[2] * a[2]) + a[3] * a[3]);
    const double E = gm1(a[4]) + ke;
    s.U[0] = a[0];
    s.U[1] = m;
    s.U[2] = a[0] * a[2];
    s.U[3] = a[0] * a[3];
    s.U[4] = E;
    s.U[5] = a[0] * a[5];
    s.F[0] = m;
    s.F[1] = m * a[1] + a[4];
    s.F[2] = m * a[2];
    s.F[3] = m * a[3];
    s.F[4] = (E + a[4]) * a[1];
    s.F[5] = s.U[5] * a[1];
}

template <bool SHORT>
__device__ __forceinline__ bool hlle_by(const double* qL, const double* qR, double gamma, double* F)
{
    Recip<SHORT> gm1(gamma - 1.0);
    const double cL = sqrt((gamma * qL[4]) / qL[0]);
    const double cR = sqrt((gamma * qR[4]) / qR[0]);
    const double a1 = qL[1] - cL, a2 = qR[1] - cR;
    const double b1 = qL[1] + cL, b2 = qR[1] + cR;
    const double SL = a1 < a2 ? a1 : a2;
    const double SR = b1 > b2 ? b1 : b2;
    const double bm = SL < 0.0 ? SL : 0.0;
    const double bp = SR > 0.0 ? SR : 0.0;
    HlleState L, R;
    hlle_side(qL, gm1, L);
    hlle_side(qR, gm1, R);
    const double bpm = bp * bm;
    Recip<SHORT> den(bp - bm);
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        const double num = (bp * L.F[v] - bm * R.F[v]) + bpm * (R.U[v] - L.U[v]);
        F[v] = den(num);
    }
    return gm1.exact() && den.exact();
}

__device__ __forceinline__ void hlle(const double* qL, const double* qR, double gamma, double* F)
{
    if (!hlle_by<true>(qL, qR, gamma, F)) hlle_by<false>(qL, qR, gamma, F);
}

// weight of the first operand of min/max in the cotangent (1, 0 or 1/2 at a tie)
__device__ __forceinline__ double wfirst_min(double a, double b) { return a < b ? 1.0 : (b < a ? 0.0 : 0.5); }
__device__ __forceinline__ double wfirst_max(double a, double b) { return a > b ? 1.0 : (b > a ? 0.0 : 0.5); }

// cotangent of one side's U and F back to its state a = (rho, u, v, w, p, Ye)
__device__ __forceinline__ void hlle_side_vjp(const double* a, Recip<>& gm1, const double* Ub,
                                              const double* Fb, double* ab)
{
    const double rho = a[0], u = a[1], v = a[2], w = a[3], p = a[4], ye = a[5];
    const double m = rho * u;
    const double v2 = (u * u + v * v) + w * w;
    const double E = gm1(p) + (0.5 * rho) * v2;
    const double mb = Ub[1] + Fb[0] + Fb[1] * u + Fb[2] * v + Fb[3] * w;
    const double Eb = Ub[4] + Fb[4] * u;
    const double U5b = Ub[5] + Fb[5] * u;
    ab[0] += Ub[0] + Ub[2] * v + Ub[3] * w + U5b * ye + mb * u + Eb * (0.5 * v2);
    ab[1] += mb * rho + Fb[1] * m + Fb[4] * (E + p) + Fb[5] * (rho * ye) + Eb * (rho * u);
    ab[2] += Ub[2] * rho + Fb[2] * m + Eb * (rho * v);
    ab[3] += Ub[3] * rho + Fb[3] * m + Eb * (rho * w);
    ab[4] += Fb[1] + Fb[4] * u + gm1(Eb);
    ab[5] += U5b * rho;
}

// HLLE VJP: given Fbar, accumulate qLbar, qRbar (rotated order)
__device__ __forceinline__ void hlle_vjp(const double* qL, const double* qR, double gamma,
                                         const double* Fb, double* qLb, double* qRb)
{
    Recip<> gm1(gamma - 1.0), rL(qL[0]), rR(qR[0]);
    const double cL = sqrt(rL(gamma * qL[4]));
    const double cR = sqrt(rR(gamma * qR[4]));
    const double a1 = qL[1] - cL, a2 = qR[1] - cR;
    const double b1 = qL[1] + cL, b2 = qR[1] + cR;
    const double SL = a1 < a2 ? a1 : a2;
    const double SR = b1 > b2 ? b1 : b2;
    const double bm = SL < 0.0 ? SL : 0.0;
    const double bp = SR > 0.0 ? SR : 0.0;
    HlleState L, R;
    hlle_side(qL, gm1, L);
    hlle_side(qR, gm1, R);
    const double bpm = bp * bm;
    const double den = bp - bm;
    double bpb = 0.0, bmb = 0.0, bpmb = 0.0, denb = 0.0;
    double ULb[6], URb[6], FLb[6], FRb[6];
    const double inv_den = 1.0 / den;
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        const double num = (bp * L.F[v] - bm * R.F[v]) + bpm * (R.U[v] - L.U[v]);
        const double F = num * inv_den;
        const double nb = Fb[v] * inv_den;
        denb -= nb * F;
        bpb += nb * L.F[v];
        bmb -= nb * R.F[v];
        bpmb += nb * (R.U[v] - L.U[v]);
        FLb[v] = nb * bp;
        FRb[v] = -nb * bm;
        URb[v] = nb * bpm;
        ULb[v] = -nb * bpm;
    }
    bpb += bpmb * bm + denb;
    bmb += bpmb * bp - denb;
    const double SRb = bpb * wfirst_max(SR, 0.0);
    const double SLb = bmb * wfirst_min(SL, 0.0);
    const double wa = wfirst_min(a1, a2), wb = wfirst_max(b1, b2);
    const double a1b = SLb * wa, a2b = SLb * (1.0 - wa);
    const double b1b = SRb * wb, b2b = SRb * (1.0 - wb);
    hlle_side_vjp(qL, gm1, ULb, FLb, qLb);
    hlle_side_vjp(qR, gm1, URb, FRb, qRb);
    // u -/+ c
    qLb[1] += a1b + b1b;
    qRb[1] += a2b + b2b;
    const double cLb = b1b - a1b, cRb = b2b - a2b;
    // c = sqrt(gamma p / rho): dc/dp = gamma / (2 c rho), dc/drho = -c / (2 rho)
    qLb[4] += cLb * (gamma / (2.0 * cL * qL[0]));
    qLb[0] -= cLb * rL(0.5 * cL);
    qRb[4] += cRb * (gamma / (2.0 * cR * qR[0]));
    qRb[0] -= cRb * rR(0.5 * cR);
}

// variable r of the face frame of direction D at a cell: rho, v_n, v_t1, v_t2,
// p, Ye; the velocity rows are picked at compile time
template <int D>
__device__ __forceinline__ void face_frame(const AdjGeom& g, const double* __restrict__ W, int64_t c,
                                           double* q)
{
    const int64_t N = g.N;
#pragma unroll
    for (int r = 0; r < 6; ++r) q[r] = W[rmap(D, r) * N + c];
    q[4] = ((g.gamma - 1.0) * q[0]) * q[4];
}

// Windows: `rows` rows of n cells, each with `halo` wrapped cells at either end,
// laid end to end and cut into windows of `width` entries that overlap by 2 halo.
// Entry `i` of window w: its row (clamped; false where there is none) and its
// position.  The outputs of a window are its entries [halo, width - halo) at
// positions [0, n).
__host__ __device__ inline unsigned window_count(unsigned rows, int n, int halo, int width)
{
    const unsigned entries = rows * (unsigned)(n + 2 * halo), step = (unsigned)(width - 2 * halo);
    return (entries + step - 1) / step;
}

__device__ __forceinline__ bool window_entry(unsigned rows, int n, int halo, int width, unsigned w,
                                             int i, unsigned& row, int& p)
{
    const unsigned len = (unsigned)(n + 2 * halo);
    const unsigned v = w * (unsigned)(width - 2 * halo) + (unsigned)i;
    const unsigned r = v / len;
    p = (int)(v - r * len) - halo;
    row = r < rows ? r : rows - 1;
    return r < rows;
}

// Windows along x (D = 0) and y (1): a workgroup has XW positions of XT pencils
// that are neighbours in memory; neighbouring positions exchange through LDS.
constexpr int XW = 32, XT = 8, NTX = XW * XT;

__host__ __device__ inline unsigned pencil_groups(const AdjGeom& g, int d)
{
    return ((unsigned)(g.N / g.n[d]) + XT - 1) / XT;
}

// This thread's entry of window w: base and stride of its pencil, its position p
// (false where it has no output), and the threads of its neighbours.
template <int D>
__device__ __forceinline__ bool pencil_entry(const AdjGeom& g, int halo, unsigned w, int64_t& base,
                                             int64_t& stride, int& p, int& tm, int& tp)
{
    const int t = threadIdx.x, i = t / XT, n = g.n[D];
    const unsigned T = (unsigned)(g.N / n), nz = (unsigned)g.n[2];
    unsigned group;
    bool out = window_entry(pencil_groups(g, D), n, halo, XW, w, i, group, p);
    unsigned item = group * XT + t % XT;
    out = out && item < T && i >= halo && i < XW - halo && p >= 0 && p < n;
    item = item < T ? item : T - 1;
    if (D == 0) {
        base = item;
        stride = T;
    } else {
        const unsigned x = item / nz;
        base = (int64_t)x * g.n[1] * nz + (item - x * nz);
        stride = nz;
    }
    tm = i > 0 ? t - XT : t;
    tp = i < XW - 1 ? t + XT : t;
    return out;
}

// Flux differences F(p + 1/2) - F(p - 1/2) along D, dF[(D 6 + v) N + c].
template <int D>
__device__ __forceinline__ void flux_window(const AdjGeom& g, double (*X)[NTX], double (*Y)[NTX],
                                            const double* __restrict__ W, double* __restrict__ dF,
                                            unsigned w)
{
    int64_t base, stride;
    int p, tm, tp;
    const bool out = pencil_entry<D>(g, 1, w, base, stride, p, tm, tp);
    const int t = threadIdx.x, n = g.n[D];
    const int64_t c = base + wrap(p, n) * stride;
    double qm[6], q[6], qp[6], L[6], R[6], F[6];
    face_frame<D>(g, W, base + wrap(p - 1, n) * stride, qm);
    face_frame<D>(g, W, c, q);
    face_frame<D>(g, W, base + wrap(p + 1, n) * stride, qp);
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        const double s = va(q[r] - qm[r], qp[r] - q[r], g.eps2);
        R[r] = q[r] - 0.5 * s;
        X[r][t] = q[r] + 0.5 * s;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 6; ++r) L[r] = X[r][tm];         // the state left of face p - 1/2
    hlle(L, R, g.gamma, F);
#pragma unroll
    for (int r = 0; r < 6; ++r) Y[r][t] = F[r];
    __syncthreads();
    if (out) {
#pragma unroll
        for (int r = 0; r < 6; ++r) dF[(D * 6 + rmap(D, r)) * g.N + c] = Y[r][tp] - F[r];
    }
}

__global__ void __launch_bounds__(NTX, 4) adj_flux_xy_kernel(AdjGeom g, unsigned xblocks,
                                                             const double* __restrict__ W,
                                                             double* __restrict__ dF)
{
    __shared__ double X[6][NTX], Y[6][NTX];
    if (blockIdx.x < xblocks) flux_window<0>(g, X, Y, W, dF, blockIdx.x);
    else flux_window<1>(g, X, Y, W, dF, blockIdx.x - xblocks);
}

__device__ __forceinline__ void cons6(const double* w, double* u)
{
    u[0] = w[0];
    u[1] = w[0] * w[1];
    u[2] = w[0] * w[2];
    u[3] = w[0] * w[3];
    const double v2 = (w[1] * w[1] + w[2] * w[2]) + w[3] * w[3];
    u[4] = w[0] * w[4] + (0.5 * w[0]) * v2;
    u[5] = w[0] * w[5];
}

template <bool SHORT>
__device__ __forceinline__ bool prim6(const double* u, double* w)
{
    Recip<SHORT> r(u[0]);
    w[0] = u[0];
    w[1] = r(u[1]);
    w[2] = r(u[2]);
    w[3] = r(u[3]);
    const double m2 = (u[1] * u[1] + u[2] * u[2]) + u[3] * u[3];
    w[4] = r(u[4] - r(0.5 * m2));
    w[5] = r(u[5]);
    return r.exact();
}

// The z direction and the update of a forward stage.  Wave w of the launch has
// window w of the rows (x, y).
template <int STAGE>
__global__ void __launch_bounds__(NT, 4) adj_stage_kernel(AdjGeom g, double dt,
                                                          const double* __restrict__ Win,
                                                          const double* W0,
                                                          const double* __restrict__ dF,
                                                          double* Wout)
{
    const int64_t N = g.N;
    const int lane = threadIdx.x & 63, nz = g.n[2];
    const unsigned rows = (unsigned)(N / nz);
    const unsigned w = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    if (w >= window_count(rows, nz, 1, 64)) return;        // uniform over the wave
    unsigned row;
    int z;
    bool out = window_entry(rows, nz, 1, 64, w, lane, row, z);
    out = out && lane >= 1 && lane <= 62 && z >= 0 && z < nz;
    const int64_t r0 = (int64_t)row * nz;
    double dz[6];
    {
        double qm[6], q[6], qp[6], L[6], R[6], F[6];
        face_frame<2>(g, Win, r0 + wrap(z - 1, nz), qm);
        face_frame<2>(g, Win, r0 + wrap(z, nz), q);
        face_frame<2>(g, Win, r0 + wrap(z + 1, nz), qp);
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            const double s = va(q[r] - qm[r], qp[r] - q[r], g.eps2);
            R[r] = q[r] - 0.5 * s;
            L[r] = __shfl_up(q[r] + 0.5 * s, 1);           // the state left of face z - 1/2
        }
        hlle(L, R, g.gamma, F);
#pragma unroll
        for (int r = 0; r < 6; ++r) dz[rmap(2, r)] = __shfl_down(F[r], 1) - F[r];
    }
    if (!out) return;
    const int64_t c = r0 + z;
    double sum[6];
#pragma unroll
    for (int v = 0; v < 6; ++v)
        sum[v] = ((0.0 + g.area[0] * dF[v * N + c]) + g.area[1] * dF[(6 + v) * N + c]) +
                 g.area[2] * dz[v];

    double wc[6], u[6], u0[6], u1[6], wn[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) wc[v] = Win[v * N + c];
    cons6(wc, u);
    if (STAGE == 2) {
        double w0[6];
#pragma unroll
        for (int v = 0; v < 6; ++v) w0[v] = W0[v * N + c];
        cons6(w0, u0);
    }
    double fd[6];
    Recip<> vol(g.vol);
#pragma unroll
    for (int v = 0; v < 6; ++v) fd[v] = vol(0.0 - sum[v]);
    if (!vol.exact()) {
#pragma unroll
        for (int v = 0; v < 6; ++v) fd[v] = (0.0 - sum[v]) / g.vol;
    }
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        const double ut = u[v] + dt * fd[v];
        u1[v] = STAGE == 1 ? ut : 0.5 * u0[v] + 0.5 * ut;
    }
    if (!prim6<true>(u1, wn)) prim6<false>(u1, wn);
#pragma unroll
    for (int v = 0; v < 6; ++v) Wout[v * N + c] = wn[v];
}

// ---- reverse ---------------------------------------------------------------

// Ubar = Jprim(W)^T Wbar, W = (rho, v, eint, Ye)
__device__ __forceinline__ void jprim_t(const double* w, const double* Wb, double* Ub)
{
    const double rho = w[0], e = w[4], ye = w[5];
    const double ir = 1.0 / rho;
    const double v2 = (w[1] * w[1] + w[2] * w[2]) + w[3] * w[3];
    Ub[0] = Wb[0] + ir * (-(w[1] * Wb[1] + w[2] * Wb[2] + w[3] * Wb[3]) + (0.5 * v2 - e) * Wb[4] -
                          ye * Wb[5]);
    Ub[1] = ir * (Wb[1] - w[1] * Wb[4]);
    Ub[2] = ir * (Wb[2] - w[2] * Wb[4]);
    Ub[3] = ir * (Wb[3] - w[3] * Wb[4]);
    Ub[4] = ir * Wb[4];
    Ub[5] = ir * Wb[5];
}

// Wbar = Jcons(W)^T Ubar
__device__ __forceinline__ void jcons_t(const double* w, const double* Ub, double* Wb)
{
    const double rho = w[0], e = w[4], ye = w[5];
    const double v2 = (w[1] * w[1] + w[2] * w[2]) + w[3] * w[3];
    Wb[0] = Ub[0] + w[1] * Ub[1] + w[2] * Ub[2] + w[3] * Ub[3] + (e + 0.5 * v2) * Ub[4] + ye * Ub[5];
    Wb[1] = rho * (Ub[1] + w[1] * Ub[4]);
    Wb[2] = rho * (Ub[2] + w[2] * Ub[4]);
    Wb[3] = rho * (Ub[3] + w[3] * Ub[4]);
    Wb[4] = rho * Ub[4];
    Wb[5] = rho * Ub[5];
}

__global__ void __launch_bounds__(NT) adj_w2u_kernel(int64_t N, const double* __restrict__ W,
                                                    const double* __restrict__ Wb, double* Ub)
{
    const int64_t c = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (c >= N) return;
    double w[6], wb[6], ub[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        w[v] = W[v * N + c];
        wb[v] = Wb[v * N + c];
    }
    jprim_t(w, wb, ub);
#pragma unroll
    for (int v = 0; v < 6; ++v) Ub[v * N + c] = ub[v];
}

__global__ void __launch_bounds__(NT) adj_u2w_kernel(int64_t N, const double* __restrict__ W,
                                                    const double* __restrict__ Ub, double* Wb)
{
    const int64_t c = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (c >= N) return;
    double w[6], wb[6], ub[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        w[v] = W[v * N + c];
        ub[v] = Ub[v * N + c];
    }
    jcons_t(w, ub, wb);
#pragma unroll
    for (int v = 0; v < 6; ++v) Wb[v * N + c] = wb[v];
}

// Directional part of the reverse stage.  Per face, Fbar = k (lambda_c -
// lambda_{c-1}) with lambda = Ubar and k = coef A / vol, and the HLLE VJP gives
// the cotangents GL, GR of its face states.  Per cell i with slope Delta_i and
// qL(i+1/2) = q_i + Delta_i / 2, qR(i-1/2) = q_i - Delta_i / 2: gD_i = GL(i+1/2)
// / 2 - GR(i-1/2) / 2, a_i, b_i = gD_i times the derivatives of Delta_i by its
// two differences, and the cotangent of q_i is
//   GL(i+1/2) + GR(i-1/2) + b_{i-1} + a_i - b_i - a_{i+1}.

template <int D>
__device__ __forceinline__ void frame_ub(const AdjGeom& g, const double* __restrict__ Ub, int64_t c,
                                         double* u)
{
#pragma unroll
    for (int r = 0; r < 6; ++r) u[r] = Ub[rmap(D, r) * g.N + c];
}

// Cotangents of the cells along x (D = 0) or y (1).
template <int D>
__device__ __forceinline__ void vjp_window(const AdjGeom& g, double (*X)[NTX], double (*Y)[NTX],
                                           double (*Z)[NTX], const double* __restrict__ W,
                                           const double* __restrict__ Ub, double coef,
                                           double* __restrict__ G, unsigned w)
{
    int64_t base, stride;
    int p, tm, tp;
    const bool out = pencil_entry<D>(g, 2, w, base, stride, p, tm, tp);
    const int t = threadIdx.x, n = g.n[D];
    const int64_t cm = base + wrap(p - 1, n) * stride, c = base + wrap(p, n) * stride,
                  cp = base + wrap(p + 1, n) * stride;
    const double kf = coef * (g.area[D] / g.vol);
    double R[6], L[6], dl[6], dr[6], Fb[6], GL[6], GR[6];
    {
        double qm[6], q[6], qp[6], um[6], u[6];
        face_frame<D>(g, W, cm, qm);
        face_frame<D>(g, W, c, q);
        face_frame<D>(g, W, cp, qp);
        frame_ub<D>(g, Ub, cm, um);
        frame_ub<D>(g, Ub, c, u);
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            const double s = va_d(q[r] - qm[r], qp[r] - q[r], g.eps2, dl[r], dr[r]);
            R[r] = q[r] - 0.5 * s;
            X[r][t] = q[r] + 0.5 * s;
            Fb[r] = kf * (u[r] - um[r]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        L[r] = X[r][tm];
        GL[r] = GR[r] = 0.0;
    }
    hlle_vjp(L, R, g.gamma, Fb, GL, GR);
#pragma unroll
    for (int r = 0; r < 6; ++r) Y[r][t] = GL[r];
    __syncthreads();
    double acc[6];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        const double GLp = Y[r][tp];                       // of the face p + 1/2
        const double gD = 0.5 * GLp - 0.5 * GR[r];
        const double a = dl[r] * gD, b = dr[r] * gD;
        acc[r] = GLp + GR[r] + (a - b);
        X[r][t] = b;                                       // every read of L is done
        Z[r][t] = a;
    }
    __syncthreads();
    if (out) {
#pragma unroll
        for (int r = 0; r < 6; ++r)
            G[(D * 6 + rmap(D, r)) * g.N + c] = acc[r] + X[r][tm] - Z[r][tp];
    }
}

__global__ void __launch_bounds__(NTX, 3) adj_vjp_xy_kernel(AdjGeom g, unsigned xblocks,
                                                            const double* __restrict__ W,
                                                            const double* __restrict__ Ub,
                                                            double coef, double* __restrict__ G)
{
    __shared__ double X[6][NTX], Y[6][NTX], Z[6][NTX];
    if (blockIdx.x < xblocks) vjp_window<0>(g, X, Y, Z, W, Ub, coef, G, blockIdx.x);
    else vjp_window<1>(g, X, Y, Z, W, Ub, coef, G, blockIdx.x - xblocks);
}

// The z direction, then per cell the three directions' cotangents of q = (rho, v,
// p, Ye), Wbar (p = (gamma-1) rho eint) and Ubar_out = a A + b B + Jprim(W)^T Wbar.
__global__ void __launch_bounds__(NT, 3) adj_vjp_z_kernel(AdjGeom g, const double* __restrict__ W,
                                                          const double* __restrict__ Ub,
                                                          double coef,
                                                          const double* __restrict__ G, double a,
                                                          const double* A, double b,
                                                          const double* B, double* Uout)
{
    const int lane = threadIdx.x & 63, nz = g.n[2];
    const int64_t N = g.N;
    const unsigned rows = (unsigned)(N / nz);
    const unsigned win = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    if (win >= window_count(rows, nz, 2, 64)) return;        // uniform over the wave
    unsigned row;
    int z;
    bool out = window_entry(rows, nz, 2, 64, win, lane, row, z);
    out = out && lane >= 2 && lane <= 61 && z >= 0 && z < nz;
    const int64_t r0 = (int64_t)row * nz, c = r0 + wrap(z, nz), cm = r0 + wrap(z - 1, nz);
    const double kf = coef * (g.area[2] / g.vol);
    double R[6], L[6], dl[6], dr[6], Fb[6], GL[6], GR[6], qb[6];
    {
        double qm[6], q[6], qp[6], um[6], u[6];
        face_frame<2>(g, W, cm, qm);
        face_frame<2>(g, W, c, q);
        face_frame<2>(g, W, r0 + wrap(z + 1, nz), qp);
        frame_ub<2>(g, Ub, cm, um);
        frame_ub<2>(g, Ub, c, u);
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            const double s = va_d(q[r] - qm[r], qp[r] - q[r], g.eps2, dl[r], dr[r]);
            R[r] = q[r] - 0.5 * s;
            L[r] = __shfl_up(q[r] + 0.5 * s, 1);
            Fb[r] = kf * (u[r] - um[r]);
            GL[r] = GR[r] = 0.0;
        }
    }
    hlle_vjp(L, R, g.gamma, Fb, GL, GR);
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        const double GLp = __shfl_down(GL[r], 1);             // of the face z + 1/2
        const double gD = 0.5 * GLp - 0.5 * GR[r];
        const double ca = dl[r] * gD, cb = dr[r] * gD;
        qb[rmap(2, r)] = GLp + GR[r] + (ca - cb) + __shfl_up(cb, 1) - __shfl_down(ca, 1);
    }
    if (!out) return;
    double w[6], wb[6], ub[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        w[v] = W[v * N + c];
        qb[v] = G[v * N + c] + G[(6 + v) * N + c] + qb[v];
    }
    const double gm1 = g.gamma - 1.0;
    wb[0] = qb[0] + (gm1 * w[4]) * qb[4];
    wb[1] = qb[1];
    wb[2] = qb[2];
    wb[3] = qb[3];
    wb[4] = (gm1 * w[0]) * qb[4];
    wb[5] = qb[5];
    jprim_t(w, wb, ub);
#pragma unroll
    for (int v = 0; v < 6; ++v) {
        double o = ub[v] + a * A[v * N + c];
        if (B) o += b * B[v * N + c];
        Uout[v * N + c] = o;
    }
}

inline dim3 grid_cells(int64_t N) { return dim3((unsigned)((N + NT - 1) / NT)); }

// workgroups of the windows along x, y (halo 1 forward, 2 reverse)
inline unsigned pencil_blocks(const AdjGeom& g, int d, int halo)
{
    return window_count(pencil_groups(g, d), g.n[d], halo, XW);
}

// workgroups of the z windows
inline dim3 grid_rows(const AdjGeom& g, int halo)
{
    const unsigned w = window_count((unsigned)(g.N / g.n[2]), g.n[2], halo, 64);
    return dim3((w + NT / 64 - 1) / (NT / 64));
}

}  // namespace

hipError_t launch_adj_stage(const AdjGeom& g, int stage, double dt, const double* Win,
                            const double* W0, double* F, double* Wout, hipStream_t s)
{
    const unsigned xb = pencil_blocks(g, 0, 1), yb = pencil_blocks(g, 1, 1);
    hipLaunchKernelGGL(adj_flux_xy_kernel, dim3(xb + yb), dim3(NTX), 0, s, g, xb, Win, F);
    if (stage == 1)
        hipLaunchKernelGGL(adj_stage_kernel<1>, grid_rows(g, 1), dim3(NT), 0, s, g, dt, Win, W0,
                           (const double*)F, Wout);
    else
        hipLaunchKernelGGL(adj_stage_kernel<2>, grid_rows(g, 1), dim3(NT), 0, s, g, dt, Win, W0,
                           (const double*)F, Wout);
    return hipGetLastError();
}

hipError_t launch_adj_w2u(const AdjGeom& g, const double* W, const double* Wb, double* Ub,
                          hipStream_t s)
{
    hipLaunchKernelGGL(adj_w2u_kernel, grid_cells(g.N), dim3(NT), 0, s, g.N, W, Wb, Ub);
    return hipGetLastError();
}

hipError_t launch_adj_u2w(const AdjGeom& g, const double* W, const double* Ub, double* Wb,
                          hipStream_t s)
{
    hipLaunchKernelGGL(adj_u2w_kernel, grid_cells(g.N), dim3(NT), 0, s, g.N, W, Ub, Wb);
    return hipGetLastError();
}

// Reverse of one stage with input W: Uout = a A + b B + Jprim(W)^T dL(W)^T (coef Ub);
// G: 12 N scratch.
static hipError_t reverse_stage(const AdjGeom& g, const double* W, const double* Ub, double coef,
                                double* G, double a, const double* A, double b, const double* B,
                                double* Uout, hipStream_t s)
{
    const unsigned xb = pencil_blocks(g, 0, 2), yb = pencil_blocks(g, 1, 2);
    hipLaunchKernelGGL(adj_vjp_xy_kernel, dim3(xb + yb), dim3(NTX), 0, s, g, xb, W, Ub, coef, G);
    hipLaunchKernelGGL(adj_vjp_z_kernel, grid_rows(g, 2), dim3(NT), 0, s, g, W, Ub, coef,
                       (const double*)G, a, A, b, B, Uout);
    return hipGetLastError();
}

// One reverse RK2 step: W0, W1 the stage inputs of the step, U2b the cotangent
// of its output (conserved form, overwritten by that of W0), U1b and G scratch.
hipError_t launch_adj_step_reverse(const AdjGeom& g, double dt, const double* W0, const double* W1,
                                   double* U2b, double* U1b, double* G, hipStream_t s)
{
    // stage 2: U1b = 1/2 U2b + Jprim(W1)^T dL(W1)^T (dt/2 U2b)
    if (hipError_t e = reverse_stage(g, W1, U2b, 0.5 * dt, G, 0.5, U2b, 0.0, nullptr, U1b, s)) return e;
    // stage 1: U0b = 1/2 U2b + U1b + Jprim(W0)^T dL(W0)^T (dt U1b), into U2b
    return reverse_stage(g, W0, U1b, dt, G, 0.5, U2b, 1.0, U1b, U2b, s);
}

}  // namespace fx
