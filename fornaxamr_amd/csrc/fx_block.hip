// Per-block flux assembly in the reference's own block layouts: the drop-in
// form of prj_flux_update (src/prj_flux.c:2149-2521) and prj_flux_div
// (src/prj_flux.c:2523-2533) for blocks kept in the reference's 20^3 storage.
//
// Block layouts (src/prj_defs.h:383-459, 16^3 active cells, 2 ghost layers,
// AoSoA lane width 4):
//   LIDX(i,j,k)        = ((i+2)*20 + (j+2))*20 + (k+2)
//   BIDX(nc,v,i,j,k)   = ((((i+2)*20 + (j+2))*5 + (k+2)/4)*nc + v)*4 + (k+2)%4
//   FACE_IDX(dir,...)  = LIDX with 21 slots along dir
// Faces written (src/prj_flux.c:2221-2262): normal index 0..16 in every
// direction; transverse 0..15 for hydro, -1..16 for MHD (CT needs one more
// layer).  A face (i,j,k) of direction dir lies between cell (i,j,k) - e_dir
// (left) and (i,j,k) (right).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>

#include "../../include/fornax_gpu.h"
#include "fx_kernels.hpp"
#include "fx_physics.hpp"

namespace fx {
namespace {

constexpr int NT = 256;
constexpr int RB = 20;          // reference block edge incl. ghosts (PRJ_BS)
constexpr int RNG = 2;          // ghost layers
constexpr int AW = 4;           // AoSoA lane width (PRJ_AOSOA_W)

__device__ __forceinline__ int lidx(int i, int j, int k)
{
    return ((i + RNG) * RB + (j + RNG)) * RB + (k + RNG);
}

__device__ __forceinline__ int bidx(int nc, int v, int i, int j, int k)
{
    return ((((i + RNG) * RB + (j + RNG)) * (RB / AW) + (k + RNG) / AW) * nc + v) * AW +
           (k + RNG) % AW;
}

__device__ __forceinline__ int face_idx(int dir, int i, int j, int k)
{
    if (dir == 0) return ((i + RNG) * RB + (j + RNG)) * RB + (k + RNG);
    if (dir == 1) return ((i + RNG) * (RB + 1) + (j + RNG)) * RB + (k + RNG);
    return ((i + RNG) * RB + (j + RNG)) * (RB + 1) + (k + RNG);
}

// The hydro face outputs of one wave (4 rows of 16 faces) leave through a
// wave-private LDS tile: written [row][var][k] by the computing lanes, read
// back as 16-byte pairs (k, k+1) of one variable in the arrays' own order
// (AoSoA group, variable, slot pair), so that a wave stores each row's
// 16 x 6 fluxes as 48 16-byte pieces in increasing address order (3 store
// instructions per face for the fluxes, 2 for the face velocities) where each
// variable's per-lane store scattered over ~20 cache lines.  A row's first and
// last AoSoA group hold two active k (slots 2-3 and 0-1); the ghost slots are
// not written.  Row pitches 112 / 48 doubles put the two rows of a half-wave
// in complementary LDS banks.
constexpr int SFP = 112;   // flux tile row pitch (6 x 16 + 16)
constexpr int SVP = 48;    // face-velocity tile row pitch (3 x 16)

// Piece w (0 .. 8 nc - 1, in address order) of one row of an AoSoA array of
// nc variables over the 16 active k: its variable and the first k of its pair.
__device__ __forceinline__ void row_piece(int nc, int w, int& v, int& k0)
{
    if (w < nc) {                    // group 0: slots 2-3 = k 0, 1
        v = w;
        k0 = 0;
    } else if (w < 7 * nc) {         // groups 1..3: slot pairs 0-1 and 2-3
        const int t = w - nc;
        const int g = 1 + t / (2 * nc);
        const int rem = t % (2 * nc);
        v = rem >> 1;
        k0 = 4 * g - 2 + 2 * (rem & 1);
    } else {                         // group 4: slots 0-1 = k 14, 15
        v = w - 7 * nc;
        k0 = 14;
    }
}

// Hydro: every face of a block from one pass over its cells.  A workgroup marches
// x-planes like the mesh path's stage (fx_hydro.hip): thread (j, k) owns a
// column, plane i (20 x 20 cells with their halo, 7 quantities; v1 in a ring of
// four planes) is in LDS, and per plane each thread solves the low-side x-, y-
// and z-face of its cell while half of one wave, rotating, solves the 32
// high-side y/z faces.  The face states come from the four cells along the
// normal; along x from the column's own registers.
//
// Bound: the loads and stores of the AoSoA arrays.  With x/y pencils and a
// z-face kernel every direction read W and eosvar again (64 load instructions
// per cell against 24 here, 11.5 GB against 7.7 GB for 4096 blocks).
//
// One barrier per plane.  Iteration n (plane i) reads plane i (stored before the
// barrier of n - 1) with its neighbours, plane i + 1 at its own column only, and
// v1 of planes i - 1 .. i + 1.  Plane i + 2, prefetched in registers, goes into
// plane i's slot after the barrier of n, its v1 into the ring (over plane
// i - 2) before it.  The x-face i needs velocity differences of planes i - 1
// and i: those of i - 1 were taken when it was the current plane.
struct BlockLds {
    double pl[2][7][RB * RB];            // rho v2 v3 e ye P gamma of planes i, i + 1
    double v1[4][RB * RB];               // v1 of plane p in v1[(p - x0 + 4) & 3]
    __align__(16) double f[NT / 64][4 * SFP];   // output tiles of the waves
    __align__(16) double v[NT / 64][4 * SVP];
};

__global__ void __launch_bounds__(NT, 2) block_march_kernel(const fx_block_io* __restrict__ blocks,
                                                            int split)
{
    __shared__ BlockLds L;
    constexpr int PC = RB * RB;
    constexpr int NQ = 8;                // rho v1 v2 v3 e ye P gamma
    const int t = threadIdx.x;
    const int j = t >> 4, k = t & 15;
    const int lane = t & 63, wave = t >> 6;
    // neighbouring parts of a block on one XCD (workgroups go round the 8 XCDs)
    const int nwg = gridDim.x;
    const int wg = (nwg & 7) == 0 ? (int)(blockIdx.x & 7) * (nwg >> 3) + (int)(blockIdx.x >> 3)
                                  : (int)blockIdx.x;
    const fx_block_io* bp = blocks + wg / split;
    const int np = BS / split;
    const int x0 = (wg % split) * np;
    const int x1 = x0 + np == BS ? BS + 1 : x0 + np;   // the last part adds x-face 16
    // faces x0 .. x1 - 1 need the cells of planes x0 - 2 .. x1
    const int64_t vs = bp->var_stride;
    const double* __restrict__ W = as_global(bp->W);
    const double* __restrict__ eos = as_global(bp->eosvar);

    // own cell and (t < 144) one halo cell of the 20 x 20 plane
    const int oidx = (j + RNG) * RB + (k + RNG);
    const bool has_halo = t < PC - BS * BS;
    int hj, hk;
    if (t < 80) {
        const int r = t / RB;
        hj = r < 2 ? r : r + BS;
        hk = t - r * RB;
    } else {
        const int h = t - 80, c = h & 3;
        hj = RNG + (h >> 2);
        hk = c < 2 ? c : c + BS;
    }
    const int hidx = hj * RB + hk;
    auto eidx = [](int c) { return ((c / RB) * (RB / AW) + (c % RB) / AW) * 3 * AW + (c % RB) % AW; };
    const int eo = eidx(oidx), eh = eidx(hidx);

    struct Cell { double q[NQ]; };
    auto load_cell = [&](int p, int c, int e, Cell& r) {
        // scalar plane base + 32-bit lane offset
        const double* Wp = W + (p + RNG) * PC;
        const double* Ep = eos + (p + RNG) * (PC * 3);
#pragma unroll
        for (int q = 0; q < 6; ++q) r.q[q] = at_byte(Wp + q * vs, 8u * c);
        r.q[6] = at_byte(Ep, 8u * e);
        r.q[7] = at_byte(Ep + 2 * AW, 8u * e);
    };
    auto load_plane = [&](int p, Cell& own, Cell& halo) {
        load_cell(p, oidx, eo, own);
        if (has_halo) load_cell(p, hidx, eh, halo);
    };
    auto store_cell = [&](int slot, int c, const Cell& r) {
        L.pl[slot][0][c] = r.q[0];
#pragma unroll
        for (int q = 2; q < NQ; ++q) L.pl[slot][q - 1][c] = r.q[q];
    };

    // each wave's pieces of 4 rows (i, 4 wave + r, 0..15) in the output arrays
    // and in its tile: the same for the three directions, and for every plane
    // but for its offset
    int fsrc[3], fdst[3], vsrc[2], vdst[2];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const int c = s * 64 + lane, rr = c / 48;
        int v, k0;
        row_piece(6, c % 48, v, k0);
        fsrc[s] = rr * SFP + v * 16 + k0;
        fdst[s] = bidx(6, v, 0, wave * 4 + rr, k0);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int c = s * 64 + lane, rr = (c / 24) & 3;
        int v, k0;
        row_piece(3, c % 24, v, k0);
        vsrc[s] = rr * SVP + v * 16 + k0;
        vdst[s] = bidx(3, v, 0, wave * 4 + rr, k0);
    }
    const int krow = ((lane >> 4) * SFP) + k, vrow = ((lane >> 4) * SVP) + k;
    // fluxes and face velocities of this thread's face (i, j, k) of direction dir
    auto put = [&](int dir, int i, const double* Fl, const double* vl) {
        double* F = as_global(bp->flux[dir]);
        double* vr = as_global(bp->v_riemann[dir]);
        // paired 16-byte stores where the arrays lie on 16-byte boundaries
        if (((reinterpret_cast<uintptr_t>(F) | reinterpret_cast<uintptr_t>(vr)) & 15) == 0) {
            double* sf = L.f[wave];
            double* sv = L.v[wave];
#pragma unroll
            for (int lv = 0; lv < 6; ++lv) sf[krow + gmap(dir, lv) * 16] = Fl[lv];
#pragma unroll
            for (int r = 0; r < 3; ++r) sv[vrow + (gmap(dir, 1 + r) - 1) * 16] = vl[r];
            // the tile is read by other lanes of this wave only: LDS operations
            // of a wave complete in order, the fences keep the compiler's order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            F += i * (RB * RB * 6);
            vr += i * (RB * RB * 3);
#pragma unroll
            for (int s = 0; s < 3; ++s)
                at_byte(reinterpret_cast<double2*>(F), 8u * fdst[s]) =
                    *reinterpret_cast<const double2*>(&sf[fsrc[s]]);
            at_byte(reinterpret_cast<double2*>(vr), 8u * vdst[0]) =
                *reinterpret_cast<const double2*>(&sv[vsrc[0]]);
            if (lane < 32)
                at_byte(reinterpret_cast<double2*>(vr), 8u * vdst[1]) =
                    *reinterpret_cast<const double2*>(&sv[vsrc[1]]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
#pragma unroll
            for (int lv = 0; lv < 6; ++lv) F[bidx(6, gmap(dir, lv), i, j, k)] = Fl[lv];
#pragma unroll
            for (int r = 0; r < 3; ++r) vr[bidx(3, gmap(dir, 1 + r) - 1, i, j, k)] = vl[r];
        }
    };

    Cell cm, own, halo;          // column cell i - 1; the prefetched plane
    double Ls[NQ];               // left state of x-face i
    double dy, dz;               // velocity differences of cell i - 1 (v2 along y, v3 along z)
    {
        Cell cmm, c0, h0, c1, h1;
        load_cell(x0 - 2, oidx, eo, cmm);
        load_cell(x0 - 1, oidx, eo, cm);
        const int o = (x0 - 1 + RNG) * PC;
        const double v1h = has_halo ? W[vs + o + hidx] : 0.0;
        const double v2m = W[2 * vs + o + oidx - RB], v2p = W[2 * vs + o + oidx + RB];
        const double v3m = W[3 * vs + o + oidx - 1], v3p = W[3 * vs + o + oidx + 1];
        load_plane(x0, c0, h0);
        load_plane(x0 + 1, c1, h1);
        if (x0 + 2 <= x1) load_plane(x0 + 2, own, halo);
        dy = dmin_delta(cm.q[2] - v2m, v2p - cm.q[2]);
        dz = dmin_delta(cm.q[3] - v3m, v3p - cm.q[3]);
#pragma unroll
        for (int q = 0; q < NQ; ++q) Ls[q] = cm.q[q] + mc_half(cmm.q[q], cm.q[q], c0.q[q]);
        L.v1[3][oidx] = cm.q[1];
        L.v1[0][oidx] = c0.q[1];
        L.v1[1][oidx] = c1.q[1];
        store_cell(0, oidx, c0);
        store_cell(1, oidx, c1);
        if (has_halo) {
            L.v1[3][hidx] = v1h;
            L.v1[0][hidx] = h0.q[1];
            L.v1[1][hidx] = h1.q[1];
            store_cell(0, hidx, h0);
            store_cell(1, hidx, h1);
        }
    }
    __syncthreads();

    for (int i = x0; i < x1; ++i) {
        const int n = i - x0;
        const int A = n & 1;
        const double (*P)[PC] = L.pl[A];         // plane i
        const double* Vc = L.v1[n & 3];
        // ---- x-face i (column cells i - 2 .. i + 1) ----------------------------
        {
            double c0[NQ], WL[6], WR[6], Fl[6], vl[3], pg[4];
            c0[0] = P[0][oidx];
            c0[1] = Vc[oidx];
#pragma unroll
            for (int q = 2; q < NQ; ++q) c0[q] = P[q - 1][oidx];
            const double (*N)[PC] = L.pl[A ^ 1];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const double c1 = q == 0 ? N[0][oidx] : (q == 1 ? L.v1[(n + 1) & 3][oidx] : N[q > 0 ? q - 1 : 0][oidx]);
                const double h = mc_half(cm.q[q], c0[q], c1);
                if (q < 6) {
                    WL[q] = Ls[q];
                    WR[q] = c0[q] - h;
                } else {
                    pg[2 * (q - 6)] = Ls[q];
                    pg[2 * (q - 6) + 1] = c0[q] - h;
                }
                Ls[q] = c0[q] + h;
            }
            const double* V2 = P[1];
            const double* V3 = P[2];
            const double ny = dmin_delta(c0[2] - V2[oidx - RB], V2[oidx + RB] - c0[2]);
            const double nz = dmin_delta(c0[3] - V3[oidx - 1], V3[oidx + 1] - c0[3]);
            hllc(WL, WR, pg[0], pg[1], pg[2], pg[3], c0[1] - cm.q[1], dmin_delta(dy, ny),
                 dmin_delta(dz, nz), Fl, vl);
            dy = ny;
            dz = nz;
#pragma unroll
            for (int q = 0; q < NQ; ++q) cm.q[q] = c0[q];
            put(0, i, Fl, vl);
        }
        if (i == BS) break;
        // ---- y- and z-faces of plane i: 1, 2 = own low side, 3 = high side ----------
        const double* Vm = L.v1[(n + 3) & 3];
        const double* Vp = L.v1[(n + 1) & 3];
#pragma unroll
        for (int f = 1; f <= 3; ++f) {
            if (f == 3 && !(wave == (n & 3) && lane < 32)) continue;
            int dir = f, fj = j, fk = k;
            if (f == 3) {
                dir = lane < 16 ? 1 : 2;
                fj = lane < 16 ? BS : lane - 16;
                fk = lane < 16 ? lane : BS;
            }
            const int c = (fj + RNG) * RB + (fk + RNG);
            const int S = dir == 1 ? RB : 1, T = dir == 1 ? 1 : RB;
            const int cl = c - S;
            const double* Vn = dir == 1 ? P[1] : P[2];
            const double* Vt = dir == 1 ? P[2] : P[1];
            // local order: rho, v_n, v_t1, v_t2, e, ye, P, gamma
            const double* rows[NQ] = {P[0], Vn, dir == 1 ? P[2] : Vc, dir == 1 ? Vc : P[1],
                                      P[3], P[4], P[5], P[6]};
            double WL[NQ], WR[NQ], Fl[6], vl[3];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const double* R = rows[q];
                const double s0 = R[cl - S], s1 = R[cl], s2 = R[c], s3 = R[c + S];
                WL[q] = s1 + mc_half(s0, s1, s2);
                WR[q] = s2 - mc_half(s1, s2, s3);
            }
            // velocity deltas (src/prj_flux.c:1967-2036): of the in-plane
            // transverse velocity, and of v1 along x
            const double din = dmin_delta(dmin_delta(Vt[cl] - Vt[cl - T], Vt[cl + T] - Vt[cl]),
                                          dmin_delta(Vt[c] - Vt[c - T], Vt[c + T] - Vt[c]));
            const double dx = dmin_delta(dmin_delta(Vc[cl] - Vm[cl], Vp[cl] - Vc[cl]),
                                         dmin_delta(Vc[c] - Vm[c], Vp[c] - Vc[c]));
            hllc(WL, WR, WL[6], WR[6], WL[7], WR[7], Vn[c] - Vn[cl], dir == 1 ? din : dx,
                 dir == 1 ? dx : din, Fl, vl);
            if (f < 3) {
                put(f, i, Fl, vl);
            } else {
                double* F = dir == 1 ? as_global(bp->flux[1]) : as_global(bp->flux[2]);
                double* vr = dir == 1 ? as_global(bp->v_riemann[1]) : as_global(bp->v_riemann[2]);
                const double g1 = dir == 1 ? Fl[3] : Fl[2], g2 = dir == 1 ? Fl[1] : Fl[3],
                             g3 = dir == 1 ? Fl[2] : Fl[1];
                double* Fo = F + bidx(6, 0, i, fj, fk);
                Fo[0] = Fl[0];
                Fo[AW] = g1;
                Fo[2 * AW] = g2;
                Fo[3 * AW] = g3;
                Fo[4 * AW] = Fl[4];
                Fo[5 * AW] = Fl[5];
                double* vo = vr + bidx(3, 0, i, fj, fk);
                vo[0] = dir == 1 ? vl[2] : vl[1];
                vo[AW] = dir == 1 ? vl[0] : vl[2];
                vo[2 * AW] = dir == 1 ? vl[1] : vl[0];
            }
        }
        if (i + 1 == x1) break;
        // ---- plane i + 2 -------------------------------------------------------------
        L.v1[(n + 2) & 3][oidx] = own.q[1];
        if (has_halo) L.v1[(n + 2) & 3][hidx] = halo.q[1];
        __syncthreads();
        store_cell(A, oidx, own);
        if (has_halo) store_cell(A, hidx, halo);
        if (i + 3 <= x1) load_plane(i + 3, own, halo);
    }
}

// MHD: likewise one pass over a block's cells, but the faces of a plane (the CT
// layer's included: 18 x 18 x-faces, 17 x 18 y-, 18 x 17 z-faces) are dealt to
// eight waves as 16 tasks of 64 faces of one direction, two tasks a wave: 936 of
// 1024 lanes solve a face.  Four whole planes (i - 2 .. i + 1, 11 quantities,
// 140,800 B) are in LDS, so that a face of any direction is one stencil of four
// cells and the HLLD code appears once; thread t < 400 holds cell t of the next
// plane in registers meanwhile.  One workgroup per CU, two waves per SIMD, 46-53 %
// VALU issue; sixteen waves of one task each (128 VGPRs) spilled 128 and took
// 421 us where this takes 291 (256 blocks).
//
// The planes -1 .. 16 of all blocks are dealt evenly to as many workgroups as
// there are CUs; a share that ends inside a block costs its successor the loads
// of the three planes before it, and no face is solved twice.
struct BlockMhdLds {
    double pl[4][11][RB * RB];           // rho v1 v2 v3 e ye b1 b2 b3 P gamma; plane p in slot p & 3
};
constexpr int NTM = 512;
constexpr int MP = BS + 2;               // planes -1 .. 16

__global__ void __launch_bounds__(NTM, 1) block_march_mhd_kernel(const fx_block_io* __restrict__ blocks,
                                                                 int nblocks, int* err)
{
    __shared__ BlockMhdLds L;
    constexpr int PC = RB * RB;
    constexpr int NQ = 11;
    const int t = threadIdx.x;
    const int nwg = gridDim.x;
    const int wg = (nwg & 7) == 0 ? (int)(blockIdx.x & 7) * (nwg >> 3) + (int)(blockIdx.x >> 3)
                                  : (int)blockIdx.x;
    const int64_t end = (int64_t)nblocks * MP * (wg + 1) / nwg;
    double* lds = &L.pl[0][0][0];
    const bool has_cell = t < PC;
    const int eo = ((t / RB) * (RB / AW) + (t % RB) / AW) * 3 * AW + (t % RB) % AW;

    for (int64_t at = (int64_t)nblocks * MP * wg / nwg; at < end;) {
        const fx_block_io* bp = blocks + at / MP;
        const int lo = (int)(at % MP) - 1;
        const int hi = (int)min((int64_t)(MP - 1), lo + (end - at));
        at += hi - lo;
        const int64_t vs = bp->var_stride;
        const double* __restrict__ W = as_global(bp->W);
        const double* __restrict__ eos = as_global(bp->eosvar);

        auto load_cell = [&](int p, double* q) {
            // scalar plane base + 32-bit lane offset
            const double* Wp = W + (p + RNG) * PC;
            const double* Ep = eos + (p + RNG) * (PC * 3);
#pragma unroll
            for (int v = 0; v < 9; ++v) q[v] = at_byte(Wp + v * vs, 8u * t);
            q[9] = at_byte(Ep, 8u * eo);
            q[10] = at_byte(Ep + 2 * AW, 8u * eo);
        };
        auto store_cell = [&](int p, const double* q) {
            double* s = lds + (p & 3) * (NQ * PC) + t;
#pragma unroll
            for (int v = 0; v < NQ; ++v) s[v * PC] = q[v];
        };
        if (has_cell) {
            double q[4][NQ];
#pragma unroll
            for (int p = 0; p < 4; ++p)
                if (lo - 2 + p >= -RNG) load_cell(lo - 2 + p, q[p]);
#pragma unroll
            for (int p = 0; p < 4; ++p)
                if (lo - 2 + p >= -RNG) store_cell(lo - 2 + p, q[p]);
        }
        __syncthreads();

        for (int i = lo; i < hi; ++i) {
            double nx[NQ];                   // plane i + 2
            const bool more = i + 1 < hi;
            if (more && has_cell) load_cell(i + 2, nx);
#pragma unroll 1
            for (int pass = 0; pass < 2; ++pass) {
                // tasks: 0..5 x, 6..10 y, 11..15 z
                const int task = pass * 8 + __builtin_amdgcn_readfirstlane(t >> 6);
                const int dir = task < 6 ? 0 : (task < 11 ? 1 : 2);
                const int e = (task - (dir == 0 ? 0 : (dir == 1 ? 6 : 11))) * 64 + (t & 63);
                const int w = dir == 2 ? BS + 1 : BS + 2;         // faces along k
                const int n = dir == 0 ? (BS + 2) * (BS + 2) : (BS + 1) * (BS + 2);
                if (e >= n || (dir == 0 && i < 0)) continue;
                const int j = e / w - (dir != 1), k = e - e / w * w - (dir != 2);
                const double bn = as_global(bp->bf[dir])[face_idx(dir, i, j, k)];
                const int c = (j + RNG) * RB + (k + RNG);
                const int S = dir == 1 ? RB : 1;
                const double* st[4];
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    st[s] = lds + (dir == 0 ? ((i + s + 2) & 3) * (NQ * PC) + c
                                            : (i & 3) * (NQ * PC) + c + (s - 2) * S);
                double WL[9], WR[9], pg[4];
#pragma unroll
                for (int lv = 0; lv < 9; ++lv) {
                    if (lv == B1) continue;                   // the normal field is the face value
                    const int q = gmap(dir, lv) * PC;
                    const double s0 = st[0][q], s1 = st[1][q], s2 = st[2][q], s3 = st[3][q];
                    WL[lv] = s1 + mc_half(s0, s1, s2);
                    WR[lv] = s2 - mc_half(s1, s2, s3);
                }
                WL[B1] = bn;
                WR[B1] = bn;
                // pressure and gamma reconstructed from eosvar (src/prj_flux.c:555-562)
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const int q = (9 + v) * PC;
                    const double s0 = st[0][q], s1 = st[1][q], s2 = st[2][q], s3 = st[3][q];
                    pg[2 * v] = s1 + mc_half(s0, s1, s2);
                    pg[2 * v + 1] = s2 - mc_half(s1, s2, s3);
                }
                double Fl[9], vl[3], bv1 = 0.0, bv2 = 0.0;
                const int rc = hlld<false>(WL, WR, pg[0], pg[1], pg[2], pg[3], bn, Fl, vl, &bv1, &bv2);
                if (rc != 0) {
                    if (atomicCAS(err, 0, rc) == 0) {
                        err[1] = dir;
                        err[2] = i;
                        err[3] = j;
                        err[4] = k;
                    }
                    continue;
                }
                double* F = as_global(bp->flux[dir]) + i * (PC * 9);
                const unsigned fo = 8u * bidx(9, 0, 0, j, k);
#pragma unroll
                for (int lv = 0; lv < 9; ++lv) at_byte(F + gmap(dir, lv) * AW, fo) = Fl[lv];
                double* vr = as_global(bp->v_riemann[dir]) + i * (PC * 3);
                const unsigned vo = 8u * bidx(3, 0, 0, j, k);
#pragma unroll
                for (int r = 0; r < 3; ++r) at_byte(vr + (gmap(dir, 1 + r) - 1) * AW, vo) = vl[r];
                const unsigned lo8 = 8u * lidx(0, j, k);
                at_byte(as_global(bp->Bv1[dir]) + i * PC, lo8) = bv1;
                at_byte(as_global(bp->Bv2[dir]) + i * PC, lo8) = bv2;
            }
            __syncthreads();                 // every read of plane i - 2 (and, last, of the block) done
            if (!more) break;
            if (has_cell) store_cell(i + 2, nx);
            __syncthreads();
        }
    }
}

// prj_flux_div over the active cells: out[v][i][j][k]
__global__ void __launch_bounds__(NT) block_flux_div_kernel(const double* __restrict__ f0,
                                                           const double* __restrict__ f1,
                                                           const double* __restrict__ f2,
                                                           double a0, double a1, double a2,
                                                           double vol, int nvar, double* out)
{
    const int c = blockIdx.x * NT + threadIdx.x;
    if (c >= 4096) return;
    const int k = c & 15, j = (c >> 4) & 15, i = c >> 8;
    for (int v = 0; v < nvar; ++v) {
        out[v * 4096 + c] =
            -(a0 * (f0[bidx(nvar, v, i + 1, j, k)] - f0[bidx(nvar, v, i, j, k)]) +
              a1 * (f1[bidx(nvar, v, i, j + 1, k)] - f1[bidx(nvar, v, i, j, k)]) +
              a2 * (f2[bidx(nvar, v, i, j, k + 1)] - f2[bidx(nvar, v, i, j, k)])) / vol;
    }
}

// prj_mhd_bf2bc_impl (src/prj_mhd.c:555-603) over every cell of the 20^3
// block, ghosts included: cell B = face average (the metric factor is 1 off
// GR; dividing by 1.0 is the identity).  One workgroup per block.  Cells with
// a nonzero done flag are skipped (prj_mhd_bf2bc); done == null is
// prj_mhd_bf2bc_all.  A non-finite average is not stored and is reported in
// err {1, block, i, j, k} where the reference aborts.
__global__ void __launch_bounds__(NT) block_bf2bc_kernel(const fx_bf2bc_io* __restrict__ blocks,
                                                         int* err)
{
    const fx_bf2bc_io b = blocks[blockIdx.x];
    for (int c = threadIdx.x; c < RB * RB * RB; c += NT) {
        const int k = c % RB - RNG, j = (c / RB) % RB - RNG, i = c / (RB * RB) - RNG;
        if (b.done != nullptr && b.done[c] != 0) continue;
        const double b1 = 0.5 * (b.bf[0][face_idx(0, i, j, k)] + b.bf[0][face_idx(0, i + 1, j, k)]);
        const double b2 = 0.5 * (b.bf[1][face_idx(1, i, j, k)] + b.bf[1][face_idx(1, i, j + 1, k)]);
        const double b3 = 0.5 * (b.bf[2][face_idx(2, i, j, k)] + b.bf[2][face_idx(2, i, j, k + 1)]);
        if (!isfinite(b1) || !isfinite(b2) || !isfinite(b3)) {
            if (err != nullptr && atomicCAS(err, 0, 1) == 0) {
                err[1] = blockIdx.x;
                err[2] = i;
                err[3] = j;
                err[4] = k;
            }
            continue;
        }
        b.W[(int64_t)B1 * b.var_stride + c] = b1;
        b.W[(int64_t)B2 * b.var_stride + c] = b2;
        b.W[(int64_t)B3 * b.var_stride + c] = b3;
    }
}

}  // namespace

hipError_t launch_block_bf2bc(const fx_bf2bc_io* blocks_dev, int n, int* err, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(block_bf2bc_kernel, dim3(n), dim3(NT), 0, s, blocks_dev, err);
    return hipGetLastError();
}

// compute units of the current device (0 if that cannot be had), asked for once
static int device_cus()
{
    static std::atomic<int> known[64];
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    ncu = known[dev].load(std::memory_order_relaxed);
    if (ncu == 0) {
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
        known[dev].store(ncu, std::memory_order_relaxed);
    }
    return ncu;
}

hipError_t launch_block_flux(const fx_block_io* blocks_dev, int n, int mhd, int* err,
                             hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int ncu = device_cus();
    if (mhd) {
        const int nwg = (int)std::min<int64_t>((int64_t)n * MP, std::max(ncu, 1));
        hipLaunchKernelGGL(block_march_mhd_kernel, dim3(nwg), dim3(NTM), 0, s, blocks_dev, n, err);
    } else {
        // The rule of the mesh stage, whose constants are not this kernel's (its stores
        // outlast a prologue): of all five splits on 21 counts from 1 to 4096 blocks its
        // choice was the fastest, or within 5 % of it, but for 400 blocks (268 us at
        // split 2; whole 249, split 8 240).  1 block 101 -> 12 us (16), 64 103 -> 30 (8),
        // 128 104 -> 61 (4), 256 154 -> 148 (2); 1000 and 4096 stay whole.
        const int split = stage_split(n, ncu);
        hipLaunchKernelGGL(block_march_kernel, dim3(n * split), dim3(NT), 0, s, blocks_dev, split);
    }
    return hipGetLastError();
}

hipError_t launch_block_flux_div(const double* f0, const double* f1, const double* f2,
                                 const double* area, double vol, int nvar, double* out,
                                 hipStream_t s)
{
    hipLaunchKernelGGL(block_flux_div_kernel, dim3(4096 / NT), dim3(NT), 0, s, f0, f1, f2,
                       area[0], area[1], area[2], vol, nvar, out);
    return hipGetLastError();
}

}  // namespace fx
