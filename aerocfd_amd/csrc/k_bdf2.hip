// BDF2 sub-iteration kernels: the per-direction scalar-diagonal line
// recurrences of crank2nd and the history shift of update_q0.
//
// Reference: sub_timeadvancement_2ndcrank.f90:7-467, main.f90:692-711.
// Each line of a family (xi lines over (j,k), eta over (i,k), zeta over
// (i,j)) is an independent forward/backward recurrence, so one thread runs
// one line; the three families run in the reference's order.
//
// Every kernel takes a range of the block table, so that one launch covers
// one block or all of them with the same code.
#include <algorithm>

#include "batch.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace acfd {

// block and linear-tile workgroup of an elementwise kernel: all blocks (map,
// kg) or block m0 alone (map null)
__device__ inline int crank_wg(const int *map, const KGrid *kg, int m0, long &wg)
{
    if (!map) {
        wg = xcd_slab(blockIdx.x, gridDim.x);
        return m0;
    }
    int bx, by, bz;
    const int m = batch_wg(map, kg, bx, by, bz);
    wg = bx;
    return m;
}

// ------------------------------------------------------------------ BDF2
// rhs of sub_timeadvancement_2ndcrank.f90:61-82 on the computed range and
// dq cleared on the ring.
__global__ void __launch_bounds__(256) k_crank_prep(const BlockRec *__restrict__ blks, const int *__restrict__ map,
                                                    const KGrid *__restrict__ kg, int m0, double *arena)
{
    long wg, n;
    const BlockRec &b = blks[crank_wg(map, kg, m0, wg)];
    const Ext e = b.e;
    const Box ring{e.is1 - 1, e.ie1 + 1, e.js1 - 1, e.je1 + 1, e.ks1 - 1, e.ke1 + 1};
    int i, j, k;
    if (!lin_node_at(e, ring, wg, i, j, k, n)) return;
    const long N = e.n;
    const double *q = arena + b.o.q, *q0 = arena + b.o.q0, *dt = arena + b.o.dt, *inv_j = arena + b.o.inv_j;
    const double *rhsi = arena + b.o.rhsi, *rhsv = arena + b.o.rhsv;
    double *rhs = arena + b.o.rhs, *dq = arena + b.o.w_dq;
    const bool inner = i >= e.is1 && i <= e.ie1 && j >= e.js1 && j <= e.je1 && k >= e.ks1 && k <= e.ke1;
    const double alph = 0.5, alph_i = 1.0 / (1.0 + alph);
#pragma unroll
    for (int v = 0; v < 5; v++) {
        dq[v * N + n] = 0.0;
        if (inner) {
            double r = rhsi[v * N + n] + rhsv[v * N + n];
            double qm1 = q0[(2 * v) * N + n], qz = q0[(2 * v + 1) * N + n];
            rhs[v * N + n] = alph_i * (r * dt[n] - ((1.0 + alph) * q[v * N + n] - (1.0 + 2.0 * alph) * qz
                                                    + (alph)*qm1) * inv_j[n]);
        }
    }
}

// what a line's recurrence reads at a node: velocity, sound speed, the metric
// row, dt and the value the family starts from (rhs or dq)
struct CrankNode {
    double u, v, w, c, m0, m1, m2, dt, b[5];
};
// what the next node of the line needs of the last one
struct CrankPrev {
    double u, v, w, c, m0, m1, m2, r, d[5];
};

__device__ inline double crank_rou(double u, double v, double w, double c, double m0, double m1, double m2)
{
    double temp = m0 * m0 + m1 * m1 + m2 * m2;
    temp = sqrt(temp);
    double cu = u * m0 + v * m1 + w * m2;
    return fabs(cu) + fabs(c * temp);
}

// a1..a5 of the neighbour (sub_timeadvancement_2ndcrank.f90:129-160)
__device__ inline void crank_terms(double *a, const CrankPrev &p, double hdv, int sgn, double gamma)
{
    double q2 = 0.5 * (p.u * p.u + p.v * p.v + p.w * p.w);
    double h = p.c * p.c / (gamma - 1.0) + q2;
    double cu = p.m0 * p.u + p.m1 * p.v + p.m2 * p.w;
    double b1 = hdv * (-cu * p.d[0] + p.m0 * p.d[1] + p.m1 * p.d[2] + p.m2 * p.d[3]);
    double b2 = hdv * (q2 * p.d[0] - p.u * p.d[1] - p.v * p.d[2] - p.w * p.d[3] + p.d[4]) * (gamma - 1.0);
    double b3 = sgn > 0 ? hdv * (cu + p.r) : hdv * (cu - p.r);
    a[0] = b1 + b3 * p.d[0];
    a[1] = b1 * p.u + b2 * p.m0 + b3 * p.d[1];
    a[2] = b1 * p.v + b2 * p.m1 + b3 * p.d[2];
    a[3] = b1 * p.w + b2 * p.m2 + b3 * p.d[3];
    a[4] = b1 * h + b2 * cu + b3 * p.d[4];
}

// the ring node before a line's first one
__device__ inline void crank_first(CrankPrev &p, const double *pri, const double *dxidx, const double *dq, long N, long n,
                                   int c0)
{
    p.u = pri[N + n]; p.v = pri[2 * N + n]; p.w = pri[3 * N + n]; p.c = pri[6 * N + n];
    p.m0 = dxidx[c0 * N + n]; p.m1 = dxidx[(c0 + 1) * N + n]; p.m2 = dxidx[(c0 + 2) * N + n];
    p.r = crank_rou(p.u, p.v, p.w, p.c, p.m0, p.m1, p.m2);
#pragma unroll
    for (int v = 0; v < 5; v++) p.d[v] = dq[v * N + n];
}

// one node of the recurrence: its dq into p.d, p moved on to it
__device__ inline void crank_node(CrankPrev &p, const CrankNode &C, int dir, double gamma)
{
    const double alph = 0.5, dts = C.dt / (1.0 + alph);
    double av[5];
    crank_terms(av, p, 0.5 * dts, dir, gamma);
    const double r = crank_rou(C.u, C.v, C.w, C.c, C.m0, C.m1, C.m2);
    const double div = 1.0 / (1.0 + dts * r);
#pragma unroll
    for (int v = 0; v < 5; v++) p.d[v] = dir > 0 ? div * (C.b[v] + av[v]) : C.b[v] - div * av[v];
    p.u = C.u; p.v = C.v; p.w = C.w; p.c = C.c;
    p.m0 = C.m0; p.m1 = C.m1; p.m2 = C.m2;
    p.r = r;
}

// One family of line recurrences (AXIS 1: eta lines over (i,k), 2: zeta
// over (i,j)), one thread per line, all blocks from m0 on in blockIdx.z.
// There are few lines (a 48^3 block has 36 wavefronts of them), so what
// bounds this is the latency of a line: the recurrence stays in registers
// and the operands of the next four nodes are loaded while four are computed
// (each node's loads used to wait behind the store of the last node's dq).
// Eight 48^3 blocks, one sub-iteration: eta 1035 -> 61 us, zeta 1158 ->
// 65 us, of which a factor of eight is the one launch for all blocks.
template <int AXIS>
__global__ void __launch_bounds__(64) k_crank_lines(const BlockRec *__restrict__ blks, int m0, double *arena,
                                                    double gamma)
{
    const BlockRec &rec = blks[m0 + blockIdx.z];
    const Ext e = rec.e;
    constexpr int ax2 = AXIS == 2 ? 1 : 2, c0 = 3 * AXIS;
    const int a = e.lo1(0) + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int b = e.lo1(ax2) + (int)blockIdx.y;
    if (a > e.hi1(0) || b > e.hi1(ax2)) return;
    const long N = e.n, st = e.stride(AXIS);
    const double *pri = arena + rec.o.pri, *dxidx = arena + rec.o.dxidx, *dt = arena + rec.o.dt;
    double *dq = arena + rec.o.w_dq;
    const int lo = e.lo1(AXIS), hi = e.hi1(AXIS);
    // node of line position x along AXIS: n0 + st x
    const long n0 = e.ix(a, AXIS == 1 ? 0 : b, AXIS == 2 ? 0 : b);
    CrankPrev p;
    // four nodes from x on in direction dir (positions beyond the line read
    // its end and are not used)
    auto load = [&](int x, int dir, CrankNode *C) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const long n = n0 + st * min(max(x + dir * t, lo), hi);
            C[t].u = pri[N + n]; C[t].v = pri[2 * N + n]; C[t].w = pri[3 * N + n]; C[t].c = pri[6 * N + n];
            C[t].m0 = dxidx[c0 * N + n]; C[t].m1 = dxidx[(c0 + 1) * N + n]; C[t].m2 = dxidx[(c0 + 2) * N + n];
            C[t].dt = dt[n];
#pragma unroll
            for (int v = 0; v < 5; v++) C[t].b[v] = dq[v * N + n];
        }
    };
    auto solve = [&](int x, int dir, int end, const CrankNode *C) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int xx = x + dir * t;
            if (dir > 0 ? xx > end : xx < end) return;
            crank_node(p, C[t], dir, gamma);
            const long n = n0 + st * xx;
#pragma unroll
            for (int v = 0; v < 5; v++) dq[v * N + n] = p.d[v];
        }
    };
    CrankNode A[4], B[4];
    // forward: eta from lo, zeta from lo+1 (:244, :360)
    const int f0 = AXIS == 2 ? lo + 1 : lo;
    crank_first(p, pri, dxidx, dq, N, n0 + st * (f0 - 1), c0);
    load(f0, 1, A);
    for (int x = f0; x <= hi; x += 8) {
        load(x + 4, 1, B);
        solve(x, 1, hi, A);
        load(x + 8, 1, A);
        solve(x + 4, 1, hi, B);
    }
    // backward: eta from hi, zeta from hi-1 (:288, :404)
    const int b0 = AXIS == 2 ? hi - 1 : hi;
    crank_first(p, pri, dxidx, dq, N, n0 + st * (b0 + 1), c0);
    load(b0, -1, A);
    for (int x = b0; x >= lo; x -= 8) {
        load(x - 4, -1, B);
        solve(x, -1, lo, A);
        load(x - 8, -1, A);
        solve(x - 4, -1, lo, B);
    }
}

// The xi family: a wavefront's 64 lines (consecutive j) are strided in
// memory, and a load by line touches 64 cache lines (eight 48^3 blocks: 301
// us).  So the wavefront reads and writes eight nodes of every line at a
// time, eight lanes a line, through LDS, the next eight in flight
// meanwhile: 138 us (before all this, 1332 us).
__global__ void __launch_bounds__(64) k_crank_xi(const BlockRec *__restrict__ blks, int m0, double *arena, double gamma)
{
    constexpr int CT = 8, kF = 13, kPad = CT + 1;
    __shared__ double buf[kF][64][kPad];
    const BlockRec &rec = blks[m0 + blockIdx.z];
    const Ext e = rec.e;
    const int ja = e.js1 + (int)blockIdx.x * 64, k = e.ks1 + (int)blockIdx.y;
    if (ja > e.je1 || k > e.ke1) return;
    const int l = threadIdx.x, lines = min(64, e.je1 - ja + 1);
    const bool mine = l < lines;
    const long N = e.n;
    const double *pri = arena + rec.o.pri, *dxidx = arena + rec.o.dxidx, *dt = arena + rec.o.dt;
    const double *rhs = arena + rec.o.rhs;
    double *dq = arena + rec.o.w_dq;
    const int lo = e.is1, hi = e.ie1;
    const long nl = e.ix(0, ja, k), sj = e.ni;
    auto field = [&](int f, const double *src) {
        return f < 3 ? pri + (f + 1) * N : f == 3 ? pri + 6 * N : f < 7 ? dxidx + (f - 4) * N : f == 7 ? dt
               : src + (f - 8) * N;
    };
    const int ii = l % CT;
    double g[kF][CT];
    // nodes x .. x + 7 of the lines, clamped to the lines and to the box
    auto load = [&](int x, const double *src) {
#pragma unroll
        for (int f = 0; f < kF; f++) {
            const double *s = field(f, src);
#pragma unroll
            for (int m = 0; m < CT; m++)
                g[f][m] = s[nl + sj * min(l / CT + m * (64 / CT), lines - 1) + min(max(x + ii, lo), hi)];
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int f = 0; f < kF; f++)
#pragma unroll
            for (int m = 0; m < CT; m++) buf[f][l / CT + m * (64 / CT)][ii] = g[f][m];
        __syncthreads();
    };
    CrankPrev p;
    auto chunk = [&](int x, int dir) {
        for (int t = 0; t < CT; t++) {
            const int pos = dir > 0 ? t : CT - 1 - t, xx = x + pos;
            if (xx < lo || xx > hi) continue;
            CrankNode C;
            C.u = buf[0][l][pos]; C.v = buf[1][l][pos]; C.w = buf[2][l][pos]; C.c = buf[3][l][pos];
            C.m0 = buf[4][l][pos]; C.m1 = buf[5][l][pos]; C.m2 = buf[6][l][pos]; C.dt = buf[7][l][pos];
#pragma unroll
            for (int v = 0; v < 5; v++) C.b[v] = buf[8 + v][l][pos];
            crank_node(p, C, dir, gamma);
#pragma unroll
            for (int v = 0; v < 5; v++) buf[8 + v][l][pos] = p.d[v];
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 5; v++)
#pragma unroll
            for (int m = 0; m < CT; m++) {
                const int line = l / CT + m * (64 / CT);
                if (line < lines && x + ii >= lo && x + ii <= hi) dq[v * N + nl + sj * line + x + ii] = buf[8 + v][line][ii];
            }
        __syncthreads();
    };
    const long me = nl + sj * (mine ? l : 0);
    crank_first(p, pri, dxidx, dq, N, me + lo - 1, 0);
    load(lo, rhs);
    for (int x = lo; x <= hi; x += CT) {
        stage();
        load(x + CT, rhs);
        chunk(x, 1);
    }
    // the backward pass reads what other lanes of the wavefront stored
    __threadfence_block();
    __syncthreads();
    crank_first(p, pri, dxidx, dq, N, me + hi + 1, 0);
    load(hi - CT + 1, dq);
    for (int x = hi - CT + 1; x + CT - 1 >= lo; x -= CT) {
        stage();
        load(x - CT, dq);
        chunk(x, -1);
    }
}

// q += dq / inv_j (:455-461)
__global__ void __launch_bounds__(256) k_crank_update(const BlockRec *__restrict__ blks, const int *__restrict__ map,
                                                      const KGrid *__restrict__ kg, int m0, double *arena)
{
    long wg, n;
    const BlockRec &b = blks[crank_wg(map, kg, m0, wg)];
    const Ext e = b.e;
    int i, j, k;
    if (!lin_node_at(e, Box{e.is1, e.ie1, e.js1, e.je1, e.ks1, e.ke1}, wg, i, j, k, n)) return;
    const long N = e.n;
    double *q = arena + b.o.q;
    const double *dq = arena + b.o.w_dq;
    const double ij = arena[b.o.inv_j + n];
#pragma unroll
    for (int x = 0; x < 5; x++) q[x * N + n] = q[x * N + n] + dq[x * N + n] / ij;
}

// update_q0 on the physical range (main.f90:701-708)
__global__ void __launch_bounds__(256) k_update_q0(const BlockRec *__restrict__ blks, const int *__restrict__ map,
                                                   const KGrid *__restrict__ kg, int m0, double *arena)
{
    long wg, n;
    const BlockRec &b = blks[crank_wg(map, kg, m0, wg)];
    const Ext e = b.e;
    int i, j, k;
    if (!lin_node_at(e, Box{e.is0, e.ie0, e.js0, e.je0, e.ks0, e.ke0}, wg, i, j, k, n)) return;
    const long N = e.n;
    double *q0 = arena + b.o.q0;
    const double *q = arena + b.o.q;
#pragma unroll
    for (int v = 0; v < 5; v++) {
        q0[(2 * v) * N + n] = q0[(2 * v + 1) * N + n];
        q0[(2 * v + 1) * N + n] = q[v * N + n];
    }
}

// exts: the ranges of blocks m0 .. m0 + nblk - 1; bg: the linear-tile grid
// of all blocks (null: one block)
int launch_crank(hipStream_t s, const BlockRec *blks, int m0, int nblk, const Ext *const *exts, const BatchGrid *bg,
                 double *arena, const Consts &c)
{
    if (!blks) return (int)hipErrorInvalidValue;
    int L[3] = {0, 0, 0};
    for (int m = 0; m < nblk; m++)
        for (int x = 0; x < 3; x++) L[x] = std::max(L[x], exts[m]->hi1(x) - exts[m]->lo1(x) + 1);
    if (L[0] <= 0 || L[1] <= 0 || L[2] <= 0) return 0;
    const int *map = bg ? bg->map : nullptr;
    const KGrid *kg = bg ? bg->kg : nullptr;
    const dim3 lin = bg ? dim3((unsigned)bg->total) : lin_grid(*exts[0]), nt(64, 4, 1);
    hipLaunchKernelGGL(k_crank_prep, lin, nt, 0, s, blks, map, kg, m0, arena);
    hipLaunchKernelGGL(k_crank_xi, dim3((L[1] + 63) / 64, L[2], nblk), dim3(64), 0, s, blks, m0, arena, c.gamma);
    hipLaunchKernelGGL((k_crank_lines<1>), dim3((L[0] + 63) / 64, L[2], nblk), dim3(64), 0, s, blks, m0, arena, c.gamma);
    hipLaunchKernelGGL((k_crank_lines<2>), dim3((L[0] + 63) / 64, L[1], nblk), dim3(64), 0, s, blks, m0, arena, c.gamma);
    hipLaunchKernelGGL(k_crank_update, lin, nt, 0, s, blks, map, kg, m0, arena);
    ACFD_CHECK_LAUNCH();
    return 0;
}

int launch_update_q0(hipStream_t s, const BlockRec *blks, int m0, const Ext &e, const BatchGrid *bg, double *arena)
{
    if (!blks) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_update_q0, bg ? dim3((unsigned)bg->total) : lin_grid(e), dim3(64, 4, 1), 0, s, blks,
                       bg ? bg->map : nullptr, bg ? bg->kg : nullptr, m0, arena);
    ACFD_CHECK_LAUNCH();
    return 0;
}

}  // namespace acfd
