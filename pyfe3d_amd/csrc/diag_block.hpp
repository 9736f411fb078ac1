// Pieces shared by the direct solvers (banded.hip, dissect.hip): the 32-column
// panel width, lane broadcasts and the Cholesky factorisation of a panel's
// diagonal block by one wave.
#pragma once
#include <hip/hip_runtime.h>

namespace band {

constexpr int NF = 32;   // factor panel width
constexpr int NH = NF / 2;  // diagonal block: columns per lane
typedef double v4d __attribute__((ext_vector_type(4)));

// value of x in lane l (l uniform across the wave), as a scalar broadcast
__device__ __forceinline__ double readlane_d(double x, int l)
{
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)v, l);
    const int hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// The jn x jn diagonal block held in P rows 0 .. 31, factorised in place
// by one wave (L11 and the reciprocal pivots dinv; *failed set on a
// non-positive pivot).  Lane (h, r) = (lane / 32, lane % 32) holds columns
// 16 h .. 16 h + 15 of row r.  Step k takes the pivot by readlane and
// broadcasts the multipliers L[r][k], k < r < jn, through LDS (zero
// elsewhere, two buffers so step k + 1 never overwrites what step k reads);
// the rank-1 update then runs on all 16 columns without masks: the lower
// triangle gets exactly its terms, the upper triangle and rows past jn hold
// values that are never broadcast.
__device__ __forceinline__ void diag_block(double (*P)[NF + 1], double *dinv, double (*Lk)[NF],
                                           int jn, int lane, bool &failed)
{
    int r = lane & 31, h = lane >> 5;
    // opaque per call, so the per-step lane masks and column offsets below
    // are formed where they are used instead of being kept live across
    // panels
    asm volatile("" : "+v"(r), "+v"(h));
    double l[NH];
#pragma unroll
    for (int i = 0; i < NH; i++) l[i] = P[r][NH * h + i];
#pragma unroll
    for (int k = 0; k < NF; k++) {
        if (k < jn) {
            const int kh = k / NH, ki = k % NH;
            const double d = readlane_d(l[ki], 32 * kh + k);
            if (!(d > 0.)) failed = true;
            const double sq = d > 0. ? sqrt(d) : 1.;
            const double inv = 1. / sq;
            if (h == kh) {
                l[ki] = r == k ? sq : l[ki] * inv;
                Lk[k & 1][r] = (r > k && r < jn) ? l[ki] : 0.;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            const double lr = Lk[k & 1][r];
#pragma unroll
            for (int i = 0; i < NH; i++) l[i] -= lr * Lk[k & 1][NH * h + i];
        }
    }
    // rows jn .. 31 exist in P only when jn = 32; the upper
    // triangle of the block is never read
#pragma unroll
    for (int i = 0; i < NH; i++) P[r][NH * h + i] = l[i];
    double dg = 1.;
#pragma unroll
    for (int i = 0; i < NH; i++)
        if (NH * h + i == r) dg = l[i];
    if (r < jn && (r >> 4) == h) dinv[r] = 1. / dg;
}

}  // namespace band
