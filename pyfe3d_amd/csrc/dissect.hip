// Direct solves by nested dissection: multifrontal Cholesky of many
// independent SPD systems (the diagonal blocks of a block-diagonal 6x6 BSR
// matrix), the counterpart of the reference callers' scipy spsolve
// (tests/test_quad4_static_point_load.py:84-102).
//
// Against the banded factorisation (banded.hip: one workgroup walks a plate
// 32 columns at a time, n b^2 operations in a chain of n / 32 panels) the
// separators of a plate need 2-4 times fewer operations (64 x 48 elements
// 2.4, 64 x 64 3.6, 512 plates of 8 to 64 a side 2.0) and leave a chain of
// 39 and 47 panels (64 x 48, 64 x 64), and every front of a tree level, of
// every system, is worked on at once by as many workgroups as it has row
// blocks and tiles.
//
// Per tree level (deepest first), all launches over all fronts of the level:
//   * panel p: 32 own columns of each front.  A workgroup takes 128 rows
//     below the panel's diagonal block: it forms that block (redundantly, so
//     the launch needs no exchange between workgroups) and its rows, the
//     original entries plus the children's update matrices minus the
//     products with the panels before (FP64 MFMA, operands straight from the
//     cached front), factorises the block in one wave while the others form
//     rows, and solves its rows against it;
//   * update: the front's boundary block, the children's contributions minus
//     L21 L21^T, in 64 x 64 tiles; it is read by the parent only.
// A right-hand side known at that time rides along as one more row of every
// front (its forward substitution costs no pass of its own); the triangular
// solves otherwise take one workgroup per front and level.
//
// Measured: a 64 x 48 plate (19,110 DOF) 1.04 ms to factorise and 0.33 ms for
// the backward pass, against 27.0 and 7.3 ms banded; 512 plates of 8 to 64
// elements a side (4.1e6 DOF) 17.2 + 2.1 ms against 60.8 + 6.6 ms, 118 GFLOP
// at 6.9 TFLOP/s.  The single plate is bound by its chain of 39 panel
// launches of 16-30 us (loads one behind another 6 us, the diagonal block's
// pivots 6 us, the row solve 3 us, products up to 10 us); the sweep by memory
// latency (waves wait in 65 % of their cycles) and by operands read again:
// 24 GB in the panels at 2.8 TB/s, 26 GB in the updates at 4.1 TB/s for a
// factor of 7.8 GB, the matrix cores busy in 9 % and 23 % of the cycles.
//
// Every sum has a fixed order: the same bits on every run.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include "../../include/pf3d.h"
#include "diag_block.hpp"
#include "dissect.hpp"

int pf3d_fail(int code, const char *fmt, ...);
int pf3d_hip_check(hipError_t e, const char *where);

namespace {

using namespace nd;
using band::diag_block;
using band::readlane_d;
using band::v4d;

// largest front (DOFs): its right-hand side fits LDS in the solves, and
// offsets inside it fit 32 bits
constexpr int MAX_FRONT = 6144;

// device image of a plan
struct Image {
    const Front *fronts;
    const Task *tasks;
    const int32_t *nodes, *cmap, *pnode, *ld, *rld;
    const int64_t *dest, *rdest;
};

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

struct Layout {
    size_t fronts, tasks, nodes, cmap, pnode, ld, rld, dest, rdest, total;
    explicit Layout(const Plan &p)
    {
        size_t o = 0;
        auto take = [&](size_t bytes) {
            const size_t at = o;
            o += align256(bytes);
            return at;
        };
        fronts = take(p.fronts.size() * sizeof(Front));
        tasks = take(p.tasks.size() * sizeof(Task));
        nodes = take(p.nodes.size() * 4);
        cmap = take(p.cmap.size() * 4);
        pnode = take(p.pnode.size() * 4);
        ld = take(p.ld.size() * 4);
        rld = take(p.rld.size() * 4);
        dest = take(p.dest.size() * 8);
        rdest = take(p.rdest.size() * 8);
        total = o;
    }
};

Image image_at(const Plan &p, const void *base)
{
    const Layout l(p);
    const char *b = (const char *)base;
    return Image{(const Front *)(b + l.fronts), (const Task *)(b + l.tasks),
                 (const int32_t *)(b + l.nodes), (const int32_t *)(b + l.cmap),
                 (const int32_t *)(b + l.pnode), (const int32_t *)(b + l.ld),
                 (const int32_t *)(b + l.rld), (const int64_t *)(b + l.dest),
                 (const int64_t *)(b + l.rdest)};
}

__global__ void nd_zero(int64_t n, double *__restrict__ p)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x)
        p[t] = 0.;
}

// original entries into the panels: one thread per entry of each BSR block
// on or below the diagonal of the elimination order, then (f given) one per
// entry of the right-hand side
__global__ void nd_scatter(Image g, int64_t nnzb, int64_t n_nodes, const double *__restrict__ val,
                           const double *__restrict__ f, double *__restrict__ L)
{
    const int64_t total = nnzb * 36 + (f ? 6 * n_nodes : 0);
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = t / 36;
        if (b < nnzb) {
            const int64_t d = g.dest[b];
            if (d < 0) continue;
            // consecutive lanes: consecutive rows of a column
            const int e = (int)(t - b * 36), c = e / 6, r = e - 6 * c;
            const int ld = g.ld[b];
            if (ld > 0) L[d + (int64_t)c * ld + r] = val[b * 36 + 6 * r + c];
            else L[d - (int64_t)c * ld + r] = val[b * 36 + 6 * c + r];
            continue;
        }
        const int64_t q = t - nnzb * 36, node = q / 6;
        const int d = (int)(q - 6 * node);
        L[g.rdest[node] + (int64_t)d * g.rld[node]] = f[6 * (int64_t)g.pnode[node] + d];
    }
}

// the children's update matrices as seen by one front
struct Kids {
    const double *u[2];
    int m[2], ld[2];
    const int32_t *map;  // the front's list: 2 per node
    int n;               // row of the right-hand side
};

__device__ __forceinline__ Kids kids_of(const Front *F, const Front &f, const int32_t *cmap,
                                        const double *Uc)
{
    Kids k;
    k.map = cmap + 2 * f.noff;
    k.n = f.k + f.m;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int id = c ? f.c1 : f.c0;
        k.u[c] = id < 0 ? nullptr : Uc + F[id].uoff;
        k.m[c] = id < 0 ? 0 : F[id].m;
        k.ld[c] = column(k.m[c] + 1);
    }
    return k;
}

// Tiles are computed transposed, as in the banded factorisation: lane l holds
// row r[t] (its row l % 16 of tile t) of the columns c[s][v] (column l / 16 +
// 4 v of block s), so that a load or store of a column covers 16 consecutive
// rows.  Offsets inside a front fit 32 bits (MAX_FRONT).

// acc += what the children add at (r, c).  Positions first, then every value
// of a child in one round of loads (an entry it does not have reads its
// first one and is not added).  Above the diagonal the values are arbitrary
// and must not be used.
template <int NT, int NS>
__device__ __forceinline__ void add_kids(v4d (&acc)[NT][NS], const Kids &k, const int (&r)[NT],
                                         const int (&c)[NS][4])
{
#pragma unroll
    for (int i = 0; i < 2; i++) {
        if (!k.u[i]) continue;
        int pr[NT], pc[NS][4];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int q = min(r[t], k.n - 1) / 6, p = k.map[2 * q + i];
            pr[t] = r[t] == k.n ? k.m[i] : p < 0 ? -1 : 6 * p + r[t] - 6 * q;
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int q = c[s][v] / 6, p = k.map[2 * q + i];
                pc[s][v] = p < 0 ? -1 : (6 * p + c[s][v] - 6 * q) * k.ld[i];
            }
        double x[NT][NS][4];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    x[t][s][v] = k.u[i][(pr[t] | pc[s][v]) < 0 ? 0 : pr[t] + pc[s][v]];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if ((pr[t] | pc[s][v]) >= 0) acc[t][s][v] += x[t][s][v];
    }
}

// acc -= (rows r[t]) x (rows rc[s])^T over the first kk1 columns of the
// front's panel; UN steps of four columns are loaded together, so that a
// wave waits once for UN (NT + NS) loads.
template <int NT, int NS, int UN>
__device__ __forceinline__ void tile_products(v4d (&acc)[NT][NS], const double *Lf, int ld,
                                              const int (&r)[NT], const int (&rc)[NS], int kk1,
                                              int lk)
{
    auto step = [&](const double (&a)[NS], const double (&b)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int s = 0; s < NS; s++)
                acc[t][s] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[t], acc[t][s], 0, 0, 0);
    };
    int kk = 0;
    for (; kk + 4 * UN <= kk1; kk += 4 * UN) {
        double a[UN][NS], b[UN][NT];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int o = (kk + 4 * u + lk) * ld;
#pragma unroll
            for (int s = 0; s < NS; s++) a[u][s] = -Lf[o + rc[s]];
#pragma unroll
            for (int t = 0; t < NT; t++) b[u][t] = Lf[o + r[t]];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UN; u++) step(a[u], b[u]);
    }
    for (; kk < kk1; kk += 4) {  // (own blocks of 6 x odd nodes end inside a step)
        const bool in = kk + lk < kk1;
        const int o = (in ? kk + lk : 0) * ld;
        double a[NS], b[NT];
#pragma unroll
        for (int s = 0; s < NS; s++) a[s] = in ? -Lf[o + rc[s]] : 0.;
#pragma unroll
        for (int t = 0; t < NT; t++) b[t] = in ? Lf[o + r[t]] : 0.;
        step(a, b);
    }
}

__global__ void __launch_bounds__(256, 3)
    nd_panel(Image g, int64_t task0, int p, double *__restrict__ L, double *__restrict__ D,
             const double *__restrict__ Uc, int *__restrict__ bad)
{
    __shared__ double P[RB][NF + 1];  // the workgroup's rows
    __shared__ double Q[NF][NF + 1];  // the diagonal block
    __shared__ double dinv[NF];
    __shared__ double Lk[2][NF];
    const Task task = g.tasks[task0 + blockIdx.x];
    const Front f = g.fronts[task.front];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int n = f.k + f.m, c0 = p * NF, jn = min(NF, f.k - c0);
    const int r0 = c0 + jn + task.part * RB, nr = min(RB, n + 1 - r0);
    double *Lf = L + f.loff;
    const int ld = column(n + 1), last = n;
    const Kids kids = kids_of(g.fronts, f, g.cmap, Uc);
    // (columns past the own ones repeat the last of them: not used)
    int c[2][4];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int v = 0; v < 4; v++) c[s][v] = min(c0 + 16 * s + lk + 4 * v, f.k - 1);
    const int rc[2] = {min(c0 + li, last), min(c0 + 16 + li, last)};
    bool failed = false;
    if (wave == 0) {
        // the diagonal block, formed and factorised while the other waves
        // form rows (its upper 16 x 16 tile is computed with the rest)
        v4d acc[2][2];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[t][s][v] = Lf[c[s][v] * ld + rc[t]];
        add_kids(acc, kids, rc, c);
        tile_products<2, 2, 4>(acc, Lf, ld, rc, rc, c0, lk);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    Q[16 * t + li][16 * s + lk + 4 * v] = acc[t][s][v];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        diag_block(Q, dinv, Lk, jn, lane, failed);
        if (lane >= jn && lane < NF) dinv[lane] = 0.;
    } else if (nr > 0) {
        // waves 1 .. 3 form the rows, in tiles of 16
        constexpr int NT = (RB / 16 + 2) / 3;
        v4d acc[NT][2];
        int row[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            row[t] = min(r0 + 16 * (wave - 1 + 3 * t) + li, last);
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[t][s][v] = Lf[c[s][v] * ld + row[t]];
        }
        add_kids(acc, kids, row, c);
        tile_products<NT, 2, 4>(acc, Lf, ld, row, rc, c0, lk);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int q = 16 * (wave - 1 + 3 * t) + li;
            if (q < RB)
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int v = 0; v < 4; v++) P[q][16 * s + lk + 4 * v] = acc[t][s][v];
        }
    }
    __syncthreads();
    // the rows against L11: x L11^T = a, column by column
    if (tid < nr) {
        // (L11 is read from LDS where it is used, not hoisted into registers)
        asm volatile("" ::: "memory");
        double x[NF];
#pragma unroll
        for (int c = 0; c < NF; c++) x[c] = P[tid][c];
#pragma unroll
        for (int c = 0; c < NF; c++) {
            x[c] *= dinv[c];
#pragma unroll
            for (int c2 = c + 1; c2 < NF; c2++) x[c2] -= x[c] * Q[c2][c];
            __builtin_amdgcn_sched_barrier(0);
        }
        double *o = Lf + (int64_t)c0 * ld + r0 + tid;
#pragma unroll
        for (int c = 0; c < NF; c++) P[tid][c] = x[c];
        for (int c = 0; c < jn; c++) o[c * ld] = P[tid][c];
    } else if (wave == 3 && task.part == 0) {
        // the factorised diagonal block, its reciprocal pivots on the
        // diagonal (the entries in L stay: other workgroups still read them)
        double *d = D + f.doff + (int64_t)p * NF * NF;
        for (int t = lane; t < NF * NF; t += 64) {
            const int r = t >> 5, c = t & 31;
            d[t] = r == c ? dinv[r] : (r > c && r < jn) ? Q[r][c] : 0.;
        }
    }
    if (failed && lane == 0 && task.part == 0) atomicAdd(bad, 1);
}

__global__ void __launch_bounds__(256)
    nd_update(Image g, int64_t task0, const double *__restrict__ L, const double *__restrict__ Uc,
              double *__restrict__ Uo)
{
    const Task task = g.tasks[task0 + blockIdx.x];
    const Front f = g.fronts[task.front];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int I = task.part >> 16, K = task.part & 0xffff;
    const int wi = wave >> 1, wk = wave & 1;
    if (I == K && wk > wi) return;  // above the diagonal
    const int last = f.k + f.m, ld = column(last + 1);  // (last: the right-hand side)
    const int rb = TS * I + 32 * wi, cb = TS * K + 32 * wk;  // in the boundary
    if (rb > f.m || cb >= f.m) return;
    v4d acc[2][2];
    int row[2], rc[2], c[2][4];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        row[t] = min(f.k + rb + 16 * t + li, last);
        rc[t] = min(f.k + cb + 16 * t + li, last);
#pragma unroll
        for (int v = 0; v < 4; v++) c[t][v] = min(f.k + cb + 16 * t + lk + 4 * v, last - 1);
#pragma unroll
        for (int s = 0; s < 2; s++) acc[t][s] = v4d{0., 0., 0., 0.};
    }
    add_kids(acc, kids_of(g.fronts, f, g.cmap, Uc), row, c);
    tile_products<2, 2, 4>(acc, L + f.loff, ld, row, rc, f.k, lk);
    double *U = Uo + f.uoff;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int r = rb + 16 * t + li;
        if (r > f.m) continue;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int q = cb + 16 * s + lk + 4 * v;
                if (q < f.m && r >= q) U[q * column(f.m + 1) + r] = acc[t][s][v];
            }
    }
}

// one front's part of L y = f in LDS: the own entries of v (k + m of them)
// against L11, their products subtracted from the boundary entries; T is
// scratch.  Starts and ends with a barrier.
__device__ __forceinline__ void forward_front(const Front &f, const double *Lf,
                                              const double *__restrict__ D, double *v,
                                              double (*T)[NF + 1])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = f.k + f.m;
    const int64_t ld = column(n + 1);
    for (int c0 = 0, p = 0; c0 < f.k; c0 += NF, p++) {
        const int jn = min(NF, f.k - c0);
        const double *d = D + f.doff + (int64_t)p * NF * NF;
        for (int t = tid; t < NF * NF; t += 256) T[t >> 5][t & 31] = d[t];
        __syncthreads();
        if (wave == 0) {
            double yc = lane < jn ? v[c0 + lane] : 0.;
            const int rr = lane & 31;
            for (int c = 0; c < jn; c++) {
                if (lane == c) yc *= T[c][c];
                const double yv = readlane_d(yc, c);
                if (lane > c && lane < jn) yc -= T[rr][c] * yv;
            }
            if (lane < jn) v[c0 + lane] = yc;
        }
        __syncthreads();
        for (int r = c0 + jn + tid; r < n; r += 256) {
            const double *a = Lf + (int64_t)c0 * ld + r;
            double acc = 0.;
            if (jn == NF) {
#pragma unroll 16
                for (int c = 0; c < NF; c++) acc = fma(a[(int64_t)c * ld], v[c0 + c], acc);
            } else {
#pragma unroll 6
                for (int c = 0; c < jn; c++) acc = fma(a[(int64_t)c * ld], v[c0 + c], acc);
            }
            v[r] -= acc;
        }
        __syncthreads();
    }
    if (f.k == 0) __syncthreads();
}

// one front's part of L^T x = y: the own entries of v, its boundary entries
// known; part is scratch, after_forward: T still holds the last panel's block.
// Starts and ends with a barrier.
__device__ __forceinline__ void backward_front(const Front &f, const double *Lf,
                                               const double *__restrict__ D, double *v,
                                               double (*T)[NF + 1], double *part,
                                               bool after_forward)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = f.k + f.m;
    const int64_t ld = column(n + 1);
    __syncthreads();
    for (int p = (f.k + NF - 1) / NF - 1; p >= 0; p--) {
        const int c0 = p * NF, jn = min(NF, f.k - c0);
        const double *d = D + f.doff + (int64_t)p * NF * NF;
        const bool last = c0 + jn == f.k, below = c0 + jn < n;
        if (!(last && after_forward))
            for (int t = tid; t < NF * NF; t += 256) T[t >> 5][t & 31] = d[t];
        if (below) {
            // wave w: columns 8 w .. 8 w + 7 of the panel against the rows below
            double s[8];
#pragma unroll
            for (int j = 0; j < 8; j++) s[j] = 0.;
            for (int r = c0 + jn + lane; r < n; r += 64) {
                const double vr = v[r];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    s[j] = fma(Lf[(int64_t)min(c0 + 8 * wave + j, f.k - 1) * ld + r], vr, s[j]);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) s[j] += __shfl_xor(s[j], o, 64);
                if (lane == 0) part[8 * wave + j] = s[j];
            }
        }
        __syncthreads();
        if (wave == 0) {
            const int rr = lane & 31;
            double rhs = lane < jn ? v[c0 + lane] - (below ? part[rr] : 0.) : 0.;
            for (int c = jn - 1; c >= 0; c--) {
                if (lane == c) rhs *= T[c][c];
                const double xv = readlane_d(rhs, c);
                if (lane < c) rhs -= T[c][rr] * xv;
            }
            if (lane < jn) v[c0 + lane] = rhs;
        }
        __syncthreads();
    }
}

// L y = f, front by front: own part of y (permuted numbering) from f and the
// children's boundary parts, then the front's own boundary part into w
__global__ void __launch_bounds__(256)
    nd_forward(Image g, int64_t front0, const double *__restrict__ L, const double *__restrict__ D,
               const double *__restrict__ f0, double *__restrict__ y, double *__restrict__ w)
{
    extern __shared__ double v[];  // k + m entries
    __shared__ double T[NF][NF + 1];
    const Front f = g.fronts[front0 + blockIdx.x];
    const int n = f.k + f.m;
    const int32_t *map = g.cmap + 2 * f.noff;
    const double *w0 = f.c0 < 0 ? nullptr : w + g.fronts[f.c0].woff;
    const double *w1 = f.c1 < 0 ? nullptr : w + g.fronts[f.c1].woff;
    for (int r = threadIdx.x; r < n; r += 256) {
        const int q = r / 6, d = r - 6 * q;
        double s = r < f.k ? f0[6 * (int64_t)g.pnode[f.own0 + q] + d] : 0.;
        if (w0 && map[2 * q] >= 0) s += w0[6 * map[2 * q] + d];
        if (w1 && map[2 * q + 1] >= 0) s += w1[6 * map[2 * q + 1] + d];
        v[r] = s;
    }
    forward_front(f, L + f.loff, D, v, T);
    for (int r = threadIdx.x; r < n; r += 256) {
        if (r < f.k) y[6 * (int64_t)f.own0 + r] = v[r];
        else w[f.woff + r - f.k] = v[r];
    }
}

// L^T x = y, parents before children; x also goes back to the original
// numbering.  fused: y is the panels' last row (the right-hand side was
// carried through the factorisation).
__global__ void __launch_bounds__(256)
    nd_backward(Image g, int64_t front0, const double *__restrict__ L,
                const double *__restrict__ D, double *__restrict__ y, double *__restrict__ x,
                int fused)
{
    extern __shared__ double v[];
    __shared__ double T[NF][NF + 1];
    __shared__ double part[NF];
    const Front f = g.fronts[front0 + blockIdx.x];
    const int n = f.k + f.m;
    const int32_t *nodes = g.nodes + f.noff;
    const double *Lf = L + f.loff;
    const int64_t ld = column(n + 1);
    for (int r = threadIdx.x; r < n; r += 256) {
        const int q = r / 6;
        v[r] = fused && r < f.k ? Lf[r * ld + n] : y[6 * (int64_t)nodes[q] + r - 6 * q];
    }
    backward_front(f, Lf, D, v, T, part, false);
    for (int r = threadIdx.x; r < f.k; r += 256) {
        const int q = r / 6, d = r - 6 * q;
        y[6 * (int64_t)f.own0 + r] = v[r];
        x[6 * (int64_t)g.pnode[f.own0 + q] + d] = v[r];
    }
}

// both passes of fronts without parents or children (a plan of one level):
// one launch, the same bits.  Plates of up to 3 x 3 elements are one front:
// 2 x 2, solved again with its factor, 133 us a call (131 by the banded
// kernel) against 139 in two launches.
__global__ void __launch_bounds__(256)
    nd_solve_alone(Image g, int64_t front0, const double *__restrict__ L,
                   const double *__restrict__ D, const double *__restrict__ f0,
                   double *__restrict__ x)
{
    extern __shared__ double v[];
    __shared__ double T[NF][NF + 1];
    __shared__ double part[NF];
    const Front f = g.fronts[front0 + blockIdx.x];
    const int32_t *pnode = g.pnode + f.own0;
    for (int r = threadIdx.x; r < f.k; r += 256) v[r] = f0[6 * (int64_t)pnode[r / 6] + r % 6];
    forward_front(f, L + f.loff, D, v, T);
    backward_front(f, L + f.loff, D, v, T, part, true);
    for (int r = threadIdx.x; r < f.k; r += 256) x[6 * (int64_t)pnode[r / 6] + r % 6] = v[r];
}

inline unsigned blocks(int64_t n, int64_t most)
{
    return (unsigned)std::min((n + 255) / 256, most);
}

// fn(first, count) over [first, last) in launches of at most 2^23 blocks (of
// 256 threads: a launch has fewer than 2^32)
template <typename F>
void in_launches(int64_t first, int64_t last, F fn)
{
    for (; first < last; first += 1 << 23)
        fn(first, dim3((unsigned)std::min(last - first, (int64_t)1 << 23)));
}

}  // namespace

extern "C" {

int pf3d_nd_create(int64_t n_nodes, const int32_t *row_ptr, const int32_t *col_idx,
                   const int32_t *coord, int64_t n_sys, const int64_t *node0, int leaf,
                   void **plan)
{
    if (n_nodes <= 0 || n_nodes > 357913941 || !row_ptr || !col_idx || n_sys <= 0 || !node0 ||
        leaf < 1 || !plan)
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: bad arguments");
    *plan = nullptr;
    if (node0[0] != 0 || node0[n_sys] != n_nodes || row_ptr[0] != 0)
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: the systems must cover the nodes");
    for (int64_t s = 0; s < n_sys; s++) {
        if (node0[s + 1] < node0[s])
            return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: node0 must not decrease");
        for (int64_t r = node0[s]; r < node0[s + 1]; r++) {
            if (row_ptr[r + 1] < row_ptr[r])
                return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: row_ptr must not decrease");
            for (int b = row_ptr[r]; b < row_ptr[r + 1]; b++)
                if (col_idx[b] < node0[s] || col_idx[b] >= node0[s + 1])
                    return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: a block couples two systems");
        }
    }
    Plan *p = nullptr;
    try {
        p = new Plan;
        build(*p, n_nodes, row_ptr, col_idx, coord, n_sys, node0, leaf);
    } catch (const std::exception &) {
        delete p;
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: out of memory");
    }
    if (p->widest > MAX_FRONT || p->fronts.size() > 2000000000 || p->tasks.size() > 2000000000) {
        const int w = p->widest;
        delete p;
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_create: a front of %d DOFs exceeds %d", w, MAX_FRONT);
    }
    *plan = p;
    return PF3D_OK;
}

int pf3d_nd_sizes(const void *plan, int64_t *sizes, double *flops)
{
    if (!plan || !sizes || !flops) return pf3d_fail(PF3D_E_ARG, "pf3d_nd_sizes: bad arguments");
    const Plan &p = *(const Plan *)plan;
    sizes[0] = (int64_t)Layout(p).total;
    sizes[1] = p.l_size + p.d_size;
    sizes[2] = p.u_size[0] + p.u_size[1];
    sizes[3] = 6 * p.n_nodes + p.w_size;
    sizes[4] = (int64_t)p.fronts.size();
    sizes[5] = p.widest;
    *flops = p.flops;
    return PF3D_OK;
}

int pf3d_nd_image(const void *plan, void *image)
{
    if (!plan || !image) return pf3d_fail(PF3D_E_ARG, "pf3d_nd_image: bad arguments");
    const Plan &p = *(const Plan *)plan;
    const Layout l(p);
    char *b = (char *)image;
    memcpy(b + l.fronts, p.fronts.data(), p.fronts.size() * sizeof(Front));
    memcpy(b + l.tasks, p.tasks.data(), p.tasks.size() * sizeof(Task));
    memcpy(b + l.nodes, p.nodes.data(), p.nodes.size() * 4);
    memcpy(b + l.cmap, p.cmap.data(), p.cmap.size() * 4);
    memcpy(b + l.pnode, p.pnode.data(), p.pnode.size() * 4);
    memcpy(b + l.ld, p.ld.data(), p.ld.size() * 4);
    memcpy(b + l.rld, p.rld.data(), p.rld.size() * 4);
    memcpy(b + l.dest, p.dest.data(), p.dest.size() * 8);
    memcpy(b + l.rdest, p.rdest.data(), p.rdest.size() * 8);
    return PF3D_OK;
}

int pf3d_nd_free(void *plan)
{
    delete (Plan *)plan;
    return PF3D_OK;
}

int pf3d_nd_factor(const void *plan, const void *image, const double *val, const double *f,
                   double *factor, double *update, int *bad, void *stream)
{
    if (!plan || !image || !val || !factor || !update || !bad)
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_factor: null argument");
    const Plan &p = *(const Plan *)plan;
    const Image g = image_at(p, image);
    hipStream_t s = (hipStream_t)stream;
    double *L = factor, *D = factor + p.l_size;
    double *U[2] = {update, update + p.u_size[0]};
    hipLaunchKernelGGL(nd_zero, dim3(blocks(p.l_size, 1 << 14)), dim3(256), 0, s, p.l_size, L);
    // (one pass up to 2^31 threads: a launch has fewer than 2^32)
    hipLaunchKernelGGL(nd_scatter, dim3(blocks(p.nnzb * 36 + (f ? 6 * p.n_nodes : 0), 1 << 23)),
                       dim3(256), 0, s, g, p.nnzb, p.n_nodes, val, f, L);
    int depth = (int)p.levels.size() - 1;
    for (const Level &lv : p.levels) {
        const double *Uc = U[(depth + 1) & 1];
        for (size_t q = 0; q < lv.panels.size(); q++) {
            in_launches(lv.panels[q].first, lv.panels[q].second, [&](int64_t t, dim3 n) {
                hipLaunchKernelGGL(nd_panel, n, dim3(256), 0, s, g, t, (int)q, L, D, Uc, bad);
            });
        }
        in_launches(lv.upd0, lv.upd1, [&](int64_t t, dim3 n) {
            hipLaunchKernelGGL(nd_update, n, dim3(256), 0, s, g, t, L, Uc, U[depth & 1]);
        });
        depth--;
    }
    return pf3d_hip_check(hipGetLastError(), "pf3d_nd_factor");
}

int pf3d_nd_solve(const void *plan, const void *image, const double *factor, const double *f,
                  double *x, double *work, void *stream)
{
    if (!plan || !image || !factor || !x || !work)
        return pf3d_fail(PF3D_E_ARG, "pf3d_nd_solve: null argument");
    const Plan &p = *(const Plan *)plan;
    const Image g = image_at(p, image);
    hipStream_t s = (hipStream_t)stream;
    const double *L = factor, *D = factor + p.l_size;
    double *y = work, *w = work + 6 * p.n_nodes;
    const size_t lds = (size_t)p.widest * sizeof(double);
    if (f && p.levels.size() == 1) {
        in_launches(p.levels[0].front0, p.levels[0].front1, [&](int64_t t, dim3 n) {
            hipLaunchKernelGGL(nd_solve_alone, n, dim3(256), lds, s, g, t, L, D, f, x);
        });
        return pf3d_hip_check(hipGetLastError(), "pf3d_nd_solve");
    }
    if (f)
        for (const Level &lv : p.levels)
            in_launches(lv.front0, lv.front1, [&](int64_t t, dim3 n) {
                hipLaunchKernelGGL(nd_forward, n, dim3(256), lds, s, g, t, L, D, f, y, w);
            });
    for (size_t i = p.levels.size(); i-- > 0;)
        in_launches(p.levels[i].front0, p.levels[i].front1, [&](int64_t t, dim3 n) {
            hipLaunchKernelGGL(nd_backward, n, dim3(256), lds, s, g, t, L, D, y, x, f ? 0 : 1);
        });
    return pf3d_hip_check(hipGetLastError(), "pf3d_nd_solve");
}

}  // extern "C"
