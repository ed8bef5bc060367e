// Host build of the library's HLLD solver (fornaxamr_amd/csrc/fx_physics.hpp) as one
// lane, compiled by tests/test_hlld_host.py once for every filling of unset
// variables.  hip_runtime.h is the empty file that the test puts in its place.
#include <cmath>
#include <cstdint>
#include <cstring>
#include <initializer_list>

using std::fmax;
using std::fmin;
using std::isfinite;

#define __host__
#define __device__
#define __forceinline__ inline
static struct {
    unsigned x;
} threadIdx, blockDim;
static void __syncthreads() {}
static double __shfl_xor(double v, int) { return v; }
static long long __double_as_longlong(double v)
{
    long long b;
    memcpy(&b, &v, 8);
    return b;
}
static double __longlong_as_double(long long b)
{
    double v;
    memcpy(&v, &b, 8);
    return v;
}
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_update_dpp(old, x, a, b, c, d) (x)
#define __builtin_amdgcn_ballot_w64(x) ((x) ? 1ull : 0ull)
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_rsq(x) (1.0 / sqrt(x))

#include "../fornaxamr_amd/csrc/fx_physics.hpp"

// n faces: W [2][n][9], p, g [2][n], bn [n]; out [n][14]: flux, face velocity, Bv1, Bv2
extern "C" void fx_test_hlld(int n, const double* W, const double* p, const double* g,
                             const double* bn, double* out, int* status)
{
    for (int i = 0; i < n; ++i) {
        double F[9], vf[3], e1, e2;
        status[i] = fx::hlld(W + 9 * i, W + 9 * (n + i), p[i], p[n + i], g[i], g[n + i], bn[i], F,
                             vf, &e1, &e2);
        double* o = out + 14 * i;
        memcpy(o, F, sizeof(F));
        memcpy(o + 9, vf, sizeof(vf));
        o[12] = e1;
        o[13] = e2;
    }
}
