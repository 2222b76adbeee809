// First-order implicit update: the LU-SGS sweeps of implicit1st.
//
// Reference: sub_timeadvancement_jac.f90:7-63 (calc_jm) and
// sub_timeadvancement_1stimplicit.f90:7-585 (implicit1st).
//
// LU-SGS is a lexicographic Gauss-Seidel sweep: node (i,j,k) needs dq* of
// (i-1,j,k), (i,j-1,k) and (i,j,k-1) and nothing else of the current sweep.
// Nodes on one hyperplane i+j+k = l are independent, and any schedule that
// respects these three dependencies computes every node from the same
// operands as the sequential loop.  Two schedules:
//
//   hyperplanes  one launch per plane l (2 (Li+Lj+Lk-2) launches per step),
//                operands read in place.
//
//   tiles        one persistent launch per sweep.  Each workgroup owns an
//                8 x 8 tile of (j,k) lines and marches along i on a skewed
//                clock: lane (tj,tk) handles the node at sweep position
//                s - tj - tk at step s.
//                * Sweep layout.  Before the forward sweep the operands of
//                  every node (metric rows, 1/J, q, sound speed, the time
//                  term phi/dt, rhs: 22 values; the sweeps form the spectral
//                  radii and the diagonal from them) are gathered into an
//                  array ordered by (tile, step, field pair, lane), so at
//                  every step a tile reads 11 contiguous rows of 64
//                  16-byte pairs -- fully coalesced, where
//                  the natural layout would have every lane on its own cache
//                  line.  The sweeps write dq* and dq over the rhs slots and a
//                  final pass adds dq to q.
//                * Push form.  A node, once solved, forms the three
//                  off-diagonal products 1/2 inv_j (A(q; grad xi_d) +- r_d I) dq
//                  that its successors need, with its own operands: the i
//                  product stays in registers, the j and k products go to the
//                  next lanes, and the tile's last row/column hand them to
//                  the neighbouring tile through exchange slots.
//                  Each product is the same expression of the same operands
//                  as in the pull form, so both schedules give the same bits.
//                * Exchange.  Slots live in uncached memory and hold a
//                  sentinel bit pattern (a signalling NaN no arithmetic
//                  produces) until the producer stores the value; the
//                  consumer polls the value itself and writes the sentinel
//                  back.  No counters, no fences, no waits for store
//                  acknowledgements between tiles.
//
// The flux Jacobian products use the closed form of A(q) v for the Euler
// flux in generalised coordinates (one reciprocal of rho instead of the ~25
// divisions of forming calc_jm's matrix); the values agree with the matrix
// form to rounding.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "batch.hpp"
#include "common.hpp"
#include "kernels.hpp"

// No implicit contraction in this file: the sweeps' arithmetic is spelled
// out (explicit fma) so that every schedule produces the same bits.
#pragma clang fp contract(off)

namespace acfd {

// 0.5 * (A(q; m) v +- r v) * inv_j for the operands of one node
// (sub_timeadvancement_1stimplicit.f90:283-301 forward, :459-477 backward).
// A v = [ m.v_mom,
//         U v_mom + u theta + m dp,
//         a1 theta + U (dp + v5) ]
// with u = mom/rho, U = m.u, theta = m.v_mom - U v1,
// dp = (gamma-1)(|u|^2/2 v1 - u.v_mom + v5), a1 = gamma E/rho - (gamma-1)|u|^2/2.
// What depends on v is all of a sweep's serial chain; the rest of a node is
// formed once, ahead of it: LuState, LuRow and LuDiag.

// the part of a node's products that no direction changes
struct LuState {
    double u, v, w, q2h, a1, s;  // velocity, |u|^2/2, a1, inv_j/2
};
// one direction: the metric row, U and +-r
struct LuRow {
    double x, y, z, U, r;
};

__device__ inline LuState lu_state(const double *qv, double ri, double ij, double gamma)
{
    LuState t;
    t.u = qv[1] * ri;
    t.v = qv[2] * ri;
    t.w = qv[3] * ri;
    t.q2h = 0.5 * fma(t.w, t.w, fma(t.v, t.v, t.u * t.u));
    t.a1 = fma(gamma * qv[4], ri, -(gamma - 1.0) * t.q2h);
    t.s = 0.5 * ij;
    return t;
}

template <int SGN>
__device__ inline LuRow lu_row(const LuState &t, double mx, double my, double mz, double rr)
{
    return {mx, my, mz, fma(mz, t.w, fma(my, t.v, mx * t.u)), SGN > 0 ? rr : -rr};
}

// dp of a solution vector v, shared by the three directions
__device__ inline double lu_dp(const LuState &t, double gamma, const double *v)
{
    const double uv = fma(t.w, v[3], fma(t.v, v[2], t.u * v[1]));
    return (gamma - 1.0) * (fma(t.q2h, v[0], -uv) + v[4]);
}

__device__ inline void lu_product(const LuState &t, const LuRow &m, double dp, const double *v, double *out)
{
    const double mvm = fma(m.z, v[3], fma(m.y, v[2], m.x * v[1]));
    const double theta = fma(-m.U, v[0], mvm);
    out[0] = t.s * fma(m.r, v[0], mvm);
    out[1] = t.s * fma(m.r, v[1], fma(m.x, dp, fma(t.u, theta, m.U * v[1])));
    out[2] = t.s * fma(m.r, v[2], fma(m.y, dp, fma(t.v, theta, m.U * v[2])));
    out[3] = t.s * fma(m.r, v[3], fma(m.z, dp, fma(t.w, theta, m.U * v[3])));
    out[4] = t.s * fma(m.r, v[4], fma(m.U, dp + v[4], t.a1 * theta));
}

// the product with the operands of node n read from the SoA fields
template <int SGN>
__device__ inline void jac_mv(const double *__restrict__ q, const double *__restrict__ dxidx,
                              const double *__restrict__ inv_j, const double *__restrict__ rr, long N, long n,
                              int c0, double gamma, const double *v, double *out)
{
    const double qv[5] = {q[n], q[N + n], q[2 * N + n], q[3 * N + n], q[4 * N + n]};
    const LuState t = lu_state(qv, 1.0 / qv[0], inv_j[n], gamma);
    const LuRow m = lu_row<SGN>(t, dxidx[c0 * N + n], dxidx[(c0 + 1) * N + n], dxidx[(c0 + 2) * N + n], rr[n]);
    lu_product(t, m, lu_dp(t, gamma, v), v, out);
}

// A divisor known before its dividends: x / d from y = 1/d (rounded), the
// quotient estimate x y, one correction by its remainder and the division's
// own last instruction, four operations in place of a dozen.  The correction
// rounds the quotient as the division does (Markstein, IBM J. Res. Dev. 34,
// 1990), so the sweeps' results are those of the reference's two divisions,
// for a normal quotient and |x| of at least 2^-969: below that the remainder
// itself is rounded, and the quotient's last bit can differ.  v_div_fixup
// gives the quotients of infinities, zeros and NaN, which the estimate makes
// NaN (an infinite diag, of dt = 0, gives 0); without it, 2 % less time on a
// block of 33^3 and 0.6 % on 129^3.  One test a step for a NaN, and the
// divisions then, took 4 and 2 %.
struct LuDivisor {
    double d, y;
};
__device__ inline LuDivisor lu_divisor(double d) { return {d, 1.0 / d}; }
__device__ inline double lu_over(double x, const LuDivisor &b)
{
    const double q = x * b.y;
    return __builtin_amdgcn_div_fixup(fma(fma(-q, b.d, x), b.y, q), b.d, x);
}

// forward node (:345-365): dq* = (rhs + A+ dq*_i-1 + B+ dq*_j-1 + C+ dq*_k-1)/diag/inv_j
__device__ inline void lu_fwd_combine(const double *rhs, const double *ta, const double *tb, const double *tc,
                                      const LuDivisor &dg, const LuDivisor &ij, double *res)
{
#pragma unroll
    for (int x = 0; x < 5; x++) res[x] = lu_over(lu_over(rhs[x] + (ta[x] + tb[x] + tc[x]), dg), ij);
}

// backward node (:521-542): dq = dq* - (A- dq_i+1 + B- dq_j+1 + C- dq_k+1)/inv_j/diag
__device__ inline void lu_bwd_combine(const double *dqs, const double *ta, const double *tb, const double *tc,
                                      const LuDivisor &dg, const LuDivisor &ij, double *res)
{
#pragma unroll
    for (int x = 0; x < 5; x++) res[x] = dqs[x] - lu_over(lu_over(ta[x] + tb[x] + tc[x], ij), dg);
}

struct LuArgs {
    Ext e;
    const double *q, *dxidx, *inv_j, *rr, *diag, *rhs;
    double *dqs, *dq;
    double gamma;
};

__device__ inline void lu_forward(const LuArgs &a, long n, const double *vi, const double *vj,
                                  const double *vk, double *res)
{
    const long N = a.e.n, sj = a.e.ni, sk = (long)a.e.ni * a.e.nj;
    double ta[5], tb[5], tc[5], rhs[5];
    jac_mv<1>(a.q, a.dxidx, a.inv_j, a.rr, N, n - 1, 0, a.gamma, vi, ta);
    jac_mv<1>(a.q, a.dxidx, a.inv_j, a.rr + N, N, n - sj, 3, a.gamma, vj, tb);
    jac_mv<1>(a.q, a.dxidx, a.inv_j, a.rr + 2 * N, N, n - sk, 6, a.gamma, vk, tc);
#pragma unroll
    for (int x = 0; x < 5; x++) rhs[x] = a.rhs[x * N + n];
    lu_fwd_combine(rhs, ta, tb, tc, lu_divisor(a.diag[n]), lu_divisor(a.inv_j[n]), res);
}

__device__ inline void lu_backward(const LuArgs &a, long n, const double *vi, const double *vj,
                                   const double *vk, double *res)
{
    const long N = a.e.n, sj = a.e.ni, sk = (long)a.e.ni * a.e.nj;
    double ta[5], tb[5], tc[5], dqs[5];
    jac_mv<-1>(a.q, a.dxidx, a.inv_j, a.rr, N, n + 1, 0, a.gamma, vi, ta);
    jac_mv<-1>(a.q, a.dxidx, a.inv_j, a.rr + N, N, n + sj, 3, a.gamma, vj, tb);
    jac_mv<-1>(a.q, a.dxidx, a.inv_j, a.rr + 2 * N, N, n + sk, 6, a.gamma, vk, tc);
#pragma unroll
    for (int x = 0; x < 5; x++) dqs[x] = a.dqs[x * N + n];
    lu_bwd_combine(dqs, ta, tb, tc, lu_divisor(a.diag[n]), lu_divisor(a.inv_j[n]), res);
}

// rhs = rhsi + rhsv on the computed range (:72-78).  For the hyperplane
// sweeps (tiles = 0): spectral radii ra, rb, rc and diag on the ring
// is1-1..ie1+1 (:98-156), and dq* and dq cleared on the ring so that
// out-of-range neighbours read 0 (:105-106).  The tile sweeps form radii and
// diagonal themselves, and their gather the time term phi*1/dt: only rhs.
__device__ inline void lu_prep_body(const Ext &e, long wg, const double *__restrict__ pri,
                                    const double *__restrict__ dxidx, const double *__restrict__ dt,
                                    const double *__restrict__ rhsi, const double *__restrict__ rhsv,
                                    double *__restrict__ rhs, double *__restrict__ rr, double *__restrict__ diag,
                                    double *__restrict__ dqs, double *__restrict__ dq, const double *cfl,
                                    int tiles)
{
    const Box ring{e.is1 - 1, e.ie1 + 1, e.js1 - 1, e.je1 + 1, e.ks1 - 1, e.ke1 + 1};
    int i, j, k;
    long n;
    if (!lin_node_at(e, ring, wg, i, j, k, n)) return;
    const long N = e.n;
    const double phi = *cfl >= 1.0e3 ? 0.0 : 1.0;  // :98-102
    if (!tiles) diag[n] = lu_radii_diag(pri, dxidx, N, n, dt[n], phi, rr);
    bool inner = i >= e.is1 && i <= e.ie1 && j >= e.js1 && j <= e.je1 && k >= e.ks1 && k <= e.ke1;
#pragma unroll
    for (int x = 0; x < 5; x++) {
        if (!tiles) {
            dqs[x * N + n] = 0.0;
            dq[x * N + n] = 0.0;
        }
        if (inner) rhs[x * N + n] = rhsi[x * N + n] + rhsv[x * N + n];
    }
}

__global__ void __launch_bounds__(256) k_lu_prep(Ext e, const double *__restrict__ pri,
                                                 const double *__restrict__ dxidx, const double *__restrict__ dt,
                                                 const double *__restrict__ rhsi, const double *__restrict__ rhsv,
                                                 double *__restrict__ rhs, double *__restrict__ rr,
                                                 double *__restrict__ diag, double *__restrict__ dqs,
                                                 double *__restrict__ dq, const double *cfl, int tiles)
{
    lu_prep_body(e, xcd_slab(blockIdx.x, gridDim.x), pri, dxidx, dt, rhsi, rhsv, rhs, rr, diag, dqs, dq, cfl,
                 tiles);
}

// every block, for the batched tile sweeps (rhs only; dq* and dq are never
// touched); block m reads cfl[m * cfl_stride]
__global__ void __launch_bounds__(256) k_lu_prep_batch(const BlockRec *__restrict__ blks,
                                                       const int *__restrict__ map, const KGrid *__restrict__ kg,
                                                       double *arena, const double *cfl, int cfl_stride)
{
    int bx, by, bz;
    const int m = batch_wg(map, kg, bx, by, bz);
    const BlockRec &b = blks[m];
    const Ext e = b.e;
    lu_prep_body(e, bx, arena + b.o.pri, arena + b.o.dxidx, arena + b.o.dt, arena + b.o.rhsi,
                 arena + b.o.rhsv, arena + b.o.rhs, arena + b.o.w_r, arena + b.o.w_diag, arena + b.o.w_dqs,
                 arena + b.o.w_dq, cfl + (long)m * cfl_stride, 1);
}

// linear tiles of 256 nodes over the block's storage (the ring of the
// computed range is masked inside), 64 x 4 threads
dim3 lu_prep_grid(const Ext &e) { return lin_grid(e); }

int launch_lu_prep_batch(hipStream_t s, const BlockRec *blks, const BatchGrid &bg, double *arena, const double *cfl,
                         int cfl_stride)
{
    if (bg.total <= 0) return 0;
    hipLaunchKernelGGL(k_lu_prep_batch, dim3((unsigned)bg.total), dim3(64, 4, 1), 0, s, blks, bg.map, bg.kg, arena,
                       cfl, cfl_stride);
    ACFD_CHECK_LAUNCH();
    return 0;
}

// One hyperplane l of the forward (DIR = +1) or backward (DIR = -1) sweep.
// Threads cover (lj, lk) from (ja, ka); li = l - lj - lk; the backward sweep
// counts from the far corner.
template <int DIR>
__global__ void __launch_bounds__(256) k_lu_plane(LuArgs a, int l, int ja, int ka)
{
    const Ext &e = a.e;
    int lj = ja + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    int lk = ka + (int)(blockIdx.y * blockDim.y + threadIdx.y);
    int Li = e.ie1 - e.is1 + 1, Lj = e.je1 - e.js1 + 1, Lk = e.ke1 - e.ks1 + 1;
    int li = l - lj - lk;
    if (lj >= Lj || lk >= Lk || li < 0 || li >= Li) return;
    const long N = e.n, sj = e.ni, sk = (long)e.ni * e.nj;
    long n = DIR > 0 ? e.ix(e.is1 + li, e.js1 + lj, e.ks1 + lk) : e.ix(e.ie1 - li, e.je1 - lj, e.ke1 - lk);
    double *out = DIR > 0 ? a.dqs : a.dq;
    double vi[5], vj[5], vk[5], res[5];
#pragma unroll
    for (int x = 0; x < 5; x++) {
        vi[x] = out[x * N + n - DIR];
        vj[x] = out[x * N + n - DIR * sj];
        vk[x] = out[x * N + n - DIR * sk];
    }
    if (DIR > 0) lu_forward(a, n, vi, vj, vk, res);
    else lu_backward(a, n, vi, vj, vk, res);
#pragma unroll
    for (int x = 0; x < 5; x++) out[x * N + n] = res[x];
}

// q += dq on the computed range (:568-574)
__global__ void __launch_bounds__(256) k_add5(Ext e, Box b, double *__restrict__ q,
                                              const double *__restrict__ dq)
{
    int i, j, k;
    if (!box_node(b, i, j, k)) return;
    const long N = e.n;
    long n = e.ix(i, j, k);
#pragma unroll
    for (int x = 0; x < 5; x++) q[x * N + n] = q[x * N + n] + dq[x * N + n];
}

// ------------------------------------------------------------ tile sweeps
// Sweep-layout fields: dxidx 0-8, inv_j 9, q 10-14, sound speed 15, the
// time term phi/dt 16, rhs 17-21 (overwritten by dq* in the forward and dq
// in the backward sweep).  The sweeps form the spectral radii and the
// diagonal from these (lu_radius, lu_diag), with the velocity q[1..3]/q[0]
// as get_primitivevariables forms it, so the results are those of radii
// and diagonal read from the preparation pass.  The grid's operands come
// first, as whole field pairs: while the sweep layout holds the same block
// and tiling and the metrics are unchanged, a gather can leave those pairs
// in place and move only the other 12 fields.
constexpr int kSlF = 22;
constexpr int kSlQ = 10;
constexpr int kSlC = 15;
constexpr int kSlT = 16;
constexpr int kSlOut = 17;
static_assert(kSlOut % 2 == 1 && kSlOut + 5 == kSlF && kSlT == kSlOut - 1,
              "the results are the upper half of the time term's pair and the two pairs after it");
constexpr int kSlGeoPairs = 5;
// exchange sentinel: a negative signalling NaN with a payload; arithmetic
// only ever produces quiet NaNs
constexpr unsigned long long kSentinel = 0xFFF5A5A5A5A5A5A5ull;

// tile edge and lanes of a tile
constexpr int kTile = 8, kLanes = 64;

// geometry of the tiling of a block's computed range
struct SlGeom {
    int nbj, nbk, ntiles, nsteps, Li, Lj, Lk;
    long exj_tile, exk_tile;  // doubles per tile of the j / k exchange regions
    // fields are stored in pairs, so a lane's operands of one step are 11
    // 16-byte loads; double index of field f of lane l at row t
    __host__ __device__ long slot(int tile, int t, int f, int l) const {
        return ((((long)tile * nsteps + t) * (kSlF / 2) + (f >> 1)) * kLanes + l) * 2 + (f & 1);
    }
};

static SlGeom sl_geom(const Ext &e)
{
    SlGeom g;
    g.Li = e.ie1 - e.is1 + 1;
    g.Lj = e.je1 - e.js1 + 1;
    g.Lk = e.ke1 - e.ks1 + 1;
    g.nbj = (g.Lj + kTile - 1) / kTile;
    g.nbk = (g.Lk + kTile - 1) / kTile;
    g.ntiles = g.nbj * g.nbk;
    g.nsteps = g.Li + 2 * kTile - 2;
    g.exj_tile = g.exk_tile = (long)(g.Li + kTile - 1) * kTile * 5;
    return g;
}

__device__ inline unsigned long long xload_bits(const double *p)
{
    return __hip_atomic_load(reinterpret_cast<const unsigned long long *>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore_bits(double *p, unsigned long long v)
{
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The layout passes move data between the natural layout (i fastest) and
// the sweep layout through LDS.  One workgroup per tile walks the tile's
// steps in chunks of CT steps, one field pair at a time through all the
// chunks, so consecutive chunks of a line are adjacent in memory and the
// cache lines a chunk boundary splits are completed by the same workgroup
// one pair-chunk (2 CT TT doubles) later: near enough for the device-wide
// caches to return them (all pairs per chunk: 5.24 against 4.80 ms for the
// gather on the 40-block channel).  In a chunk starting at
// step t0, lane l's line contributes the CT nodes li = t0 + ii - tj - tk,
// ii = 0..CT-1, which are exactly rows t0 + ii of the sweep layout.
// Natural side: thread x handles ii = x % CT of lines x / CT + m TT/CT,
// so CT consecutive lanes touch CT consecutive doubles of one line
// (CT = kSlCt).
// Sweep side: thread x is lane x.  LDS holds [CT][TT] doubles per field
// with the line index XOR-swizzled by ii (no bank conflicts either way).
// steps a layout kernel transposes at a time
constexpr int kSlCt = 32;
// the SA return pass (one value per node) takes 16: measured 0.86 against
// 1.25 ms (the two gathers and the flow add are faster at 32)
constexpr int kSaRetCt = 16;

// node index of (tile, line, li), li in range
__device__ inline long sl_nat(const Ext &e, const SlGeom &g, int tile, int line, int li)
{
    return e.ix(e.is1 + li, e.js1 + (tile % g.nbj) * kTile + line % kTile, e.ks1 + (tile / g.nbj) * kTile + line / kTile);
}
__device__ inline bool sl_line_ok(const SlGeom &g, int tile, int line)
{
    return (tile % g.nbj) * kTile + line % kTile < g.Lj && (tile / g.nbj) * kTile + line / kTile < g.Lk;
}

// the steps [t0, t1) of part `part` of `parts` of a tile's chunks of ct steps
struct SlChunks {
    int t0, t1;
    __device__ SlChunks(int nsteps, int ct, int part, int parts)
    {
        const int n = (nsteps + ct - 1) / ct;
        t0 = n * part / parts * ct;
        t1 = min(n * (part + 1) / parts * ct, nsteps);
    }
};

// csnd: the sound speed (component 7 of pri_v); dt: of which the time term
// is formed
__device__ inline const double *gather_src(int f, long N, const double *q, const double *dxidx,
                                           const double *inv_j, const double *csnd, const double *dt,
                                           const double *rhs)
{
    return f < 9 ? dxidx + f * N : f == 9 ? inv_j : f < kSlC ? q + (f - kSlQ) * N
         : f == kSlC ? csnd : f == kSlT ? dt : rhs + (f - kSlOut) * N;
}

// phi of sub_timeadvancement_1stimplicit.f90:98-102
__device__ inline double lu_phi(const double *cfl) { return *cfl >= 1.0e3 ? 0.0 : 1.0; }

// Gather the operands of every node into the sweep layout, a field pair at
// a time (each lane then stores whole 16-byte pairs), from pair fp0 on (0:
// all kSlF fields, kSlGeoPairs: all but the grid's).
__device__ inline void sl_gather_tile(const Ext &e, const SlGeom &g, int tile, const double *__restrict__ q,
                                      const double *__restrict__ dxidx, const double *__restrict__ inv_j,
                                      const double *__restrict__ csnd, const double *__restrict__ dt,
                                      const double *cfl, const double *__restrict__ rhs, double *__restrict__ sl,
                                      int fp, int part, int parts, double *buf /* [2][CT][TT] LDS, swizzled */)
{
    constexpr int CT = kSlCt, TT = kLanes, lstep = TT / CT;
    const int x = threadIdx.x;
    const int ii_n = x % CT;
    const int tj = x % kTile, tk = x / kTile;
    const bool me_ok = sl_line_ok(g, tile, x);
    const long N = e.n;
    double2 *sl2 = reinterpret_cast<double2 *>(sl);
    const SlChunks ch(g.nsteps, CT, part, parts);
    for (int t0 = ch.t0; t0 < ch.t1; t0 += CT) {
        // natural-side node offsets of this thread's CT elements (-1: none)
        int nat[CT];  // node offsets fit 32 bits (blocks below 2^31 nodes)
#pragma unroll
        for (int m = 0; m < CT; m++) {
            const int line = m * lstep + x / CT;
            const int li = t0 + ii_n - (line % kTile) - (line / kTile);
            nat[m] = (t0 + ii_n < g.nsteps && li >= 0 && li < g.Li && sl_line_ok(g, tile, line))
                         ? (int)sl_nat(e, g, tile, line, li) : -1;
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const double *src = gather_src(2 * fp + h, N, q, dxidx, inv_j, csnd, dt, rhs);
            double v[CT];
#pragma unroll
            for (int m = 0; m < CT; m++) v[m] = nat[m] >= 0 ? src[nat[m]] : 0.0;
            if (2 * fp + h == kSlT) {
                const double phi = lu_phi(cfl);
#pragma unroll
                for (int m = 0; m < CT; m++) v[m] = nat[m] >= 0 ? phi * 1.0 / v[m] : 0.0;
            }
#pragma unroll
            for (int m = 0; m < CT; m++) {
                const int line = m * lstep + x / CT;
                buf[(h * CT + ii_n) * TT + (line ^ ii_n)] = v[m];
            }
        }
        __syncthreads();
        if (me_ok) {
#pragma unroll
            for (int ii = 0; ii < CT; ii++) {
                const int t = t0 + ii, li = t - tj - tk;
                if (t < g.nsteps && li >= 0 && li < g.Li)
                    sl2[g.slot(tile, t, 2 * fp, x) >> 1] =
                        make_double2(buf[ii * TT + (x ^ ii)], buf[(CT + ii) * TT + (x ^ ii)]);
            }
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kLanes) k_sl_gather(Ext e, SlGeom g, const double *__restrict__ q,
                                                  const double *__restrict__ dxidx,
                                                  const double *__restrict__ inv_j,
                                                  const double *__restrict__ csnd,
                                                  const double *__restrict__ dt, const double *cfl,
                                                  const double *__restrict__ rhs, double *__restrict__ sl, int fp0,
                                                  int parts)
{
    __shared__ double buf[2 * kSlCt * kLanes];
    sl_gather_tile(e, g, (int)blockIdx.x, q, dxidx, inv_j, csnd, dt, cfl, rhs, sl, fp0 + (int)blockIdx.y / parts,
                   (int)blockIdx.y % parts, parts, buf);
}

// q += dq (:568-574): the backward sweep left q + dq in the result slots of
// the sweep layout; this pass moves it to q in the natural layout, same walk
// as the gather, one field pair at a time.
__device__ inline void sl_add_tile(const Ext &e, const SlGeom &g, int tile, const double *__restrict__ sl,
                                   double *__restrict__ q, int fp, int part, int parts,
                                   double *buf /* [2][CT][TT] LDS, swizzled */)
{
    constexpr int CT = kSlCt, TT = kLanes, lstep = TT / CT;
    const int x = threadIdx.x;
    const int ii_n = x % CT;
    const int tj = x % kTile, tk = x / kTile;
    const bool me_ok = sl_line_ok(g, tile, x);
    const long N = e.n;
    const SlChunks ch(g.nsteps, CT, part, parts);
    for (int t0 = ch.t0; t0 < ch.t1; t0 += CT) {
        int nat[CT];  // node offsets fit 32 bits (blocks below 2^31 nodes)
#pragma unroll
        for (int m = 0; m < CT; m++) {
            const int line = m * lstep + x / CT;
            const int li = t0 + ii_n - (line % kTile) - (line / kTile);
            nat[m] = (t0 + ii_n < g.nsteps && li >= 0 && li < g.Li && sl_line_ok(g, tile, line))
                         ? (int)sl_nat(e, g, tile, line, li) : -1;
        }
        const int v0 = 2 * fp - kSlOut;  // component of the pair's lower field (-1: the time term)
        if (me_ok) {
            const double2 *sl2 = reinterpret_cast<const double2 *>(sl);
            double2 d[CT];
#pragma unroll
            for (int ii = 0; ii < CT; ii++) {
                const int t = t0 + ii, li = t - tj - tk;
                d[ii] = (t < g.nsteps && li >= 0 && li < g.Li) ? sl2[g.slot(tile, t, 2 * fp, x) >> 1]
                                                               : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int ii = 0; ii < CT; ii++) {
                buf[ii * TT + (x ^ ii)] = d[ii].x;
                buf[(CT + ii) * TT + (x ^ ii)] = d[ii].y;
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < CT; m++) {
            const int line = m * lstep + x / CT;
            if (nat[m] >= 0) {
                if (v0 >= 0) q[v0 * N + nat[m]] = buf[ii_n * TT + (line ^ ii_n)];
                q[(v0 + 1) * N + nat[m]] = buf[(CT + ii_n) * TT + (line ^ ii_n)];
            }
        }
        __syncthreads();
    }
}

// the results are fields 17-21: the upper half of pair 8 (whose lower half
// is the time term) and pairs 9 and 10, read as whole 16-byte pairs
__global__ void __launch_bounds__(kLanes) k_sl_add(Ext e, SlGeom g, const double *__restrict__ sl,
                                               double *__restrict__ q, int parts)
{
    __shared__ double buf[2 * kSlCt * kLanes];
    sl_add_tile(e, g, (int)blockIdx.x, sl, q, kSlOut / 2 + (int)blockIdx.y / parts, (int)blockIdx.y % parts, parts, buf);
}

// Parts of a layout pass: a workgroup takes one field pair of one tile, and
// where the tiles are few, one of `parts` runs of its chunks, so that about
// kSlWgs workgroups come together (one workgroup per tile, all pairs in
// turn, left most of the device idle).  More parts split more cache lines
// between workgroups, so a launch that has enough tiles takes one.  Gather
// before and after: 33^3 75 -> 12 us, 129^3 231 -> 114, 12 blocks of 3.2 M
// nodes 233 -> 158, 98 M nodes 4.81 -> 4.52 ms; add 129^3 114 -> 55 us; SA
// gather and return of the 12 blocks 111 -> 94 and 128 -> 60 us.
constexpr int kSlWgs = 2048;
static int sl_parts(int ntiles, int fields, int nsteps, int ct)
{
    const long wgs = (long)ntiles * fields;
    return (int)std::max(1L, std::min((long)(nsteps + ct - 1) / ct, (kSlWgs + wgs - 1) / wgs));
}

static void launch_layout(hipStream_t s, int which, const Ext &e, const SlGeom &g, const Fields &f, const LuWs &ws,
                          const double *cfl = nullptr, int fp0 = 0)
{
    const int pairs = which == 0 ? kSlF / 2 - fp0 : kSlF / 2 - kSlOut / 2;
    const int parts = sl_parts(g.ntiles, pairs, g.nsteps, kSlCt);
    const dim3 gr((unsigned)g.ntiles, (unsigned)(pairs * parts));
    if (which == 0)
        hipLaunchKernelGGL(k_sl_gather, gr, dim3(kLanes), 0, s, e, g, f.q, f.dxidx, f.inv_j, f.pri + 6 * e.n, f.dt,
                           cfl, f.rhs, ws.sl, fp0, parts);
    else
        hipLaunchKernelGGL(k_sl_add, gr, dim3(kLanes), 0, s, e, g, ws.sl, f.q, parts);
}

// Fill exchange slots with the sentinel.
__global__ void __launch_bounds__(256) k_fill_sentinel(double *p, long n)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) xstore_bits(p + i, kSentinel);
}

// The node's spectral radii and diagonal from its operands: velocity as
// get_primitivevariables forms it (sub_getpri_v.f90:39-41)
__device__ inline double lu_node_radii(const double *op, double *r)
{
    const double d = op[kSlQ];
    const double u = op[kSlQ + 1] / d, v = op[kSlQ + 2] / d, w = op[kSlQ + 3] / d;
#pragma unroll
    for (int x = 0; x < 3; x++) r[x] = lu_radius(op[3 * x], op[3 * x + 1], op[3 * x + 2], u, v, w, op[kSlC]);
    return lu_diag(op[kSlT], r);
}

// -------------------------------------------------- pipelined tile sweep
// The sweep of one 8 x 8 tile by four wavefronts that run side by side.  The
// dependency chain of a sweep is its sequence of steps (Li + Lj + Lk of
// them from corner to corner of a block, and a hop through memory at every
// tile edge), and a step done by one wavefront took 1.7 us: the operands'
// loads, the radii and diagonal (square roots, divisions) and the wait for
// the neighbours' slots all stood in the chain.  Here the chain keeps only
// what depends on the neighbours:
//   wave 0     solves: combine, three products, results out.  It reads
//              prepared operands and neighbour values from LDS a step
//              ahead; inside the tile a product passes to the next lane by
//              ds_bpermute (k, formed first) and DPP (j), so no barrier is
//              on its path.
//   preparing  step s, s + 1, ... in turn: two steps' loads in flight
//   waves      each, the state, the metric rows with their radii and the two
//              divisors with their reciprocals written to a ring of
//              kPipeRing steps.
//   last wave  fetches the j and k neighbour tiles' products from the
//              exchange slots, up to eight steps at a time, into a ring, and
//              sets the slots back to the sentinel.
// The waves meet only through counters in LDS (a wave's LDS operations
// take effect in order): the others count what is ready, wave 0 what it has
// used.  Every wait is on a wave that waits for less: preparing waves wait
// for ring space (wave 0), wave 0 for operands and for slots, the slot
// wave for the neighbouring tiles with a bounded poll; running out sets
// *err and `stop`, at which every wait of the workgroup ends.
// What bounds it: wave 0's instruction issue (about 270 instructions a step,
// of which 137 are the FP64 arithmetic, at one per four cycles or more:
// about 0.65 us a step) and 2.6 us a hop; on large batches the HBM traffic.
// Forward sweep, before (one wavefront a tile) and after: 33^3 184 -> 88 us,
// 129^3 748 -> 346, 193^3 1218 -> 740, 12 blocks of 3.2 M nodes in all
// 507 -> 350, 40 blocks of 98 M nodes 6.19 -> 6.10 ms (4.7 TB/s).  Tiles of
// 16 x 16, 16 x 8 and 16 x 4 lines of the one-wavefront form were slower at
// every one of these sizes and are gone.
// A lane with nothing to do at a step takes part with zeros, which it is
// given when the step is prepared (rho 1, every other operand 0, divisors 1
// with reciprocals 0), so that its products are zero and no lane branches.  It
// takes nothing from its row of the layout: the blocks of a context share
// the layout, and the row may hold operands of another block, NaN among them.
constexpr int kPipeRing = 4;    // steps of prepared operands in LDS
constexpr int kPipeXRing = 16;  // steps of neighbour values in LDS
constexpr int kPipePrep = 2;    // preparing waves
constexpr int kPipeThreads = 64 * (1 + kPipePrep + 1);

// a prepared step, pairs of doubles per lane: rhs 0-4 (dq* in the backward
// sweep), the divisors diag and inv_j (d, y, y, d), |u|^2/2, a1, the time
// term, then forward u, v, w, r of the i row; backward q 0-4, 1/rho, r of the
// i row, unused; then x, y, z, U of the three rows and r of the j and the k
// row
template <int DIR>
struct PipeLds {
    static constexpr int kRow0 = DIR > 0 ? 8 : 10;
    static constexpr int kPairs = kRow0 + 7;
    double2 op[kPipeRing][kPairs][64];
    double x[kPipeXRing][2][5][kTile];
    int prep[kPipePrep];  // first step each preparing wave has not finished
    int xready;           // first step whose neighbour values are not there
    int done;             // steps wave 0 has finished with
    int stop;
};

__device__ inline int lds_get(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// publish after the wave's earlier LDS operations (which take effect in
// order; the barrier is for the compiler)
__device__ inline void lds_post(int *p, int v)
{
    __asm__ volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __asm__ volatile("" ::: "memory");
}

// wait until f() >= need (or the workgroup stops); the bound, some seconds,
// is only there so that no mistake can hang the device
template <typename F>
__device__ inline int lds_wait(F f, int need, int *stop, int *err)
{
    int v = __builtin_amdgcn_readfirstlane(f());
    for (long n = 0; v < need && !__builtin_amdgcn_readfirstlane(lds_get(stop)); n++) {
        if (n > (1L << 27)) {
            atomicOr(err, 1);
            lds_post(stop, 1);
        }
        v = __builtin_amdgcn_readfirstlane(f());
    }
    __asm__ volatile("" ::: "memory");
    return v;
}

// the value of the lane one (j) or eight (k) behind in the sweep's order
template <int DIR>
__device__ inline double lane_behind_j(double v)
{
    const long long b = __double_as_longlong(v);
    constexpr int ctrl = DIR > 0 ? 0x111 : 0x101;  // row_shr:1, row_shl:1
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double lane_from(int addr, double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(addr, (int)b);
    const int hi = __builtin_amdgcn_ds_bpermute(addr, (int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// preparing wave w: steps w, w + kPipePrep, ...
template <int DIR>
__device__ inline void pipe_prepare(const SlGeom &g, int tile, int w, const double *__restrict__ sl, double gamma,
                                    PipeLds<DIR> &L, int *err)
{
    const int l = threadIdx.x & 63, tj = l % kTile, tk = l / kTile;
    const bool active = (tile % g.nbj) * kTile + tj < g.Lj && (tile / g.nbj) * kTile + tk < g.Lk;
    // row of the layout at which this lane's line starts
    const int t0 = tj + tk;
    auto row = [&](int s) { return DIR > 0 ? s : g.nsteps - 1 - s; };
    auto fetch = [&](int s, double *op) {
        const double2 *src = reinterpret_cast<const double2 *>(sl + g.slot(tile, row(min(s, g.nsteps - 1)), 0, l));
#pragma unroll
        for (int f = 0; f < kSlF / 2; f++) {
            const double2 v = src[f * 64];
            op[2 * f] = v.x;
            op[2 * f + 1] = v.y;
        }
    };
    auto prepare = [&](int s, double *op) {
        if (s >= g.nsteps) return;
        const int li = row(s) - t0;
        const bool on = active && li >= 0 && li < g.Li;
        if (!on) {
#pragma unroll
            for (int f = 0; f < kSlF; f++) op[f] = f == kSlQ ? 1.0 : 0.0;
        }
        double rad[3];
        const double ri = 1.0 / op[kSlQ];
        const LuState t = lu_state(op + kSlQ, ri, op[9], gamma);
        LuDivisor dg = lu_divisor(lu_node_radii(op, rad)), ij = lu_divisor(op[9]);
        if (!on) dg.d = ij.d = 1.0, dg.y = ij.y = 0.0;
        LuRow m[3];
#pragma unroll
        for (int d = 0; d < 3; d++) m[d] = lu_row<DIR>(t, op[3 * d], op[3 * d + 1], op[3 * d + 2], rad[d]);
        lds_wait([&] { return lds_get(&L.done); }, s - kPipeRing + 1, &L.stop, err);
        double2 *o = &L.op[s % kPipeRing][0][l];
        const double *rhs = op + kSlOut;
        o[0] = make_double2(rhs[0], rhs[1]);
        o[64] = make_double2(rhs[2], rhs[3]);
        o[2 * 64] = make_double2(rhs[4], dg.d);
        o[3 * 64] = make_double2(dg.y, ij.y);
        o[4 * 64] = make_double2(ij.d, t.q2h);
        o[5 * 64] = make_double2(t.a1, op[kSlT]);
        if (DIR > 0) {
            o[6 * 64] = make_double2(t.u, t.v);
            o[7 * 64] = make_double2(t.w, m[0].r);
        } else {
            o[6 * 64] = make_double2(op[kSlQ], op[kSlQ + 1]);
            o[7 * 64] = make_double2(op[kSlQ + 2], op[kSlQ + 3]);
            o[8 * 64] = make_double2(op[kSlQ + 4], ri);
            o[9 * 64] = make_double2(m[0].r, 0.0);
        }
        double2 *r = o + PipeLds<DIR>::kRow0 * 64;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            r[2 * d * 64] = make_double2(m[d].x, m[d].y);
            r[(2 * d + 1) * 64] = make_double2(m[d].z, m[d].U);
        }
        r[6 * 64] = make_double2(m[1].r, m[2].r);
        lds_post(&L.prep[w], s + kPipePrep);
    };
    double a[kSlF], b[kSlF];
    fetch(w, a);
    fetch(w + kPipePrep, b);
    for (int s = w; s < g.nsteps; s += 2 * kPipePrep) {
        prepare(s, a);
        fetch(s + 2 * kPipePrep, a);
        prepare(s + kPipePrep, b);
        fetch(s + 3 * kPipePrep, b);
    }
}

// last wave: the neighbour tiles' products on the j side (lanes 0-31) and
// the k side (lanes 32-63).  Lane (face, r, f) loads steps d0 + r and
// d0 + 4 + r of face line f; the leading steps whose lines have all arrived
// go to the ring.  line_ok, src: of the lane's face line (no neighbour on
// that side: false, the values are zeros).
template <int DIR>
__device__ inline void pipe_fetch(const SlGeom &g, bool line_ok, int skew, double *src, PipeLds<DIR> &L, int *err)
{
    const int l = threadIdx.x & 63, face = l >> 5, r = (l >> 3) & 3, f = l & 7;
    long spins = 0;
    for (int d0 = 0; d0 < g.nsteps;) {
        lds_wait([&] { return lds_get(&L.done); }, d0 + 8 - kPipeXRing, &L.stop, err);
        if (__builtin_amdgcn_readfirstlane(lds_get(&L.stop))) return;
        unsigned long long b[2][5];
        bool need[2], ok[2];
        double *p[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int d = d0 + 4 * h + r, pos = d - skew;
            need[h] = line_ok && pos >= 0 && pos < g.Li;
            p[h] = src + (long)(need[h] ? d : 0) * kTile * 5 + f;
#pragma unroll
            for (int x = 0; x < 5; x++) b[h][x] = xload_bits(p[h] + x * kTile);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ok[h] = true;
#pragma unroll
            for (int x = 0; x < 5; x++) ok[h] = ok[h] && b[h][x] != kSentinel;
        }
        // rows of lanes that wait, both faces: bits 8 r .. 8 r + 7
        const unsigned long long m0 = __ballot(need[0] && !ok[0]), m1 = __ballot(need[1] && !ok[1]);
        const unsigned late0 = (unsigned)m0 | (unsigned)(m0 >> 32), late1 = (unsigned)m1 | (unsigned)(m1 >> 32);
        const int n = late0 ? __builtin_ctz(late0) >> 3 : late1 ? 4 + (__builtin_ctz(late1) >> 3) : 8;
        if (n == 0) {
            spins++;
            if ((spins & 1023) == 0 &&
                (spins > (1L << 21) || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                atomicOr(err, 1);
                lds_post(&L.stop, 1);
            }
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        spins = 0;
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (4 * h + r < n) {
                double *o = &L.x[(d0 + 4 * h + r) % kPipeXRing][face][0][f];
#pragma unroll
                for (int x = 0; x < 5; x++) o[x * kTile] = need[h] ? __longlong_as_double((long long)b[h][x]) : 0.0;
                if (need[h]) {
#pragma unroll
                    for (int x = 0; x < 5; x++) xstore_bits(p[h] + x * kTile, kSentinel);
                }
            }
        d0 += n;
        lds_post(&L.xready, d0);
    }
}

// wave 0: the solve
template <int DIR>
__device__ inline void pipe_solve(const SlGeom &g, int tile, double *__restrict__ sl, double gamma, double *jout,
                                  double *kout, bool pred, bool j_succ, bool k_succ, PipeLds<DIR> &L, int *err,
                                  const Ext *e, double *__restrict__ q)
{
    const int bj = tile % g.nbj, bk = tile / g.nbj;
    const int l = threadIdx.x & 63, tj = l % kTile, tk = l / kTile;
    const int lj = bj * kTile + tj, lk = bk * kTile + tk;
    const bool active = lj < g.Lj && lk < g.Lk;
    const int sj = DIR > 0 ? tj : kTile - 1 - tj, sk = DIR > 0 ? tk : kTile - 1 - tk;
    const bool fuse_add = DIR < 0 && q != nullptr;
    const long qN = fuse_add ? e->n : 0;
    const long nat0 = fuse_add && active ? e->ix(e->is1, e->js1 + lj, e->ks1 + lk) : 0;
    const bool j_out = j_succ && sj == kTile - 1, k_out = k_succ && sk == kTile - 1;
    const int behind_k = ((l - DIR * kTile) & 63) * 4;
    double ta[5] = {0, 0, 0, 0, 0}, tb[5] = {0, 0, 0, 0, 0}, tc[5] = {0, 0, 0, 0, 0};
    constexpr int kRow0 = PipeLds<DIR>::kRow0, kRows = PipeLds<DIR>::kPairs - kRow0;
    double2 E[2][kRow0], R[2][kRows];
    double fj[5], fk[5];
    int have = 0, xhave = pred ? 0 : g.nsteps;
    const int last = g.nsteps - 1;
    // The LDS reads of a step, without a branch around any of them, so that
    // the compiler's wait counts are exact and they stay in flight.  After
    // the last step they read a slot that nobody uses.
    auto wait_ops = [&](int s) {
        if (have <= s)
            have = lds_wait([&] {
                int v = lds_get(&L.prep[0]);
                for (int w = 1; w < kPipePrep; w++) v = min(v, lds_get(&L.prep[w]));
                return v;
            }, s + 1, &L.stop, err);
    };
    auto load_state = [&](int s, double2 *O) {
        const double2 *o = &L.op[s % kPipeRing][0][l];
#pragma unroll
        for (int p = 0; p < kRow0; p++) O[p] = o[p * 64];
    };
    auto load_rows = [&](int s, double2 *O) {
        const double2 *o = &L.op[s % kPipeRing][kRow0][l];
#pragma unroll
        for (int p = 0; p < kRows; p++) O[p] = o[p * 64];
    };
    auto wait_face = [&](int s) {
        if (xhave <= s) xhave = lds_wait([&] { return lds_get(&L.xready); }, s + 1, &L.stop, err);
    };
    auto load_face = [&](int s) {
        const double *v = &L.x[s % kPipeXRing][0][0][0];
#pragma unroll
        for (int x = 0; x < 5; x++) fj[x] = v[x * kTile + tk];
#pragma unroll
        for (int x = 0; x < 5; x++) fk[x] = v[(5 + x) * kTile + tj];
    };
    double2 *dst = reinterpret_cast<double2 *>(sl + g.slot(tile, DIR > 0 ? 0 : g.nsteps - 1, kSlT, l));
    double *jo = jout - (kTile - 1) * kTile * 5 + tk, *ko = kout - (kTile - 1) * kTile * 5 + tj;
    // step s with the operands E, R, while those of the next step are read
    // into NE, NR
    auto step = [&](int s, const double2 *E, const double2 *R, double2 *NE, double2 *NR) {
        wait_ops(min(s + 1, last));
        load_state(s + 1, NE);
        const int pos = s - sj - sk;
        const bool on = active && pos >= 0 && pos < g.Li;
        const double rhs[5] = {E[0].x, E[0].y, E[1].x, E[1].y, E[2].x};
        double res[5], qv[5], pb[5], pc[5];
        LuState t;
        const LuDivisor dg{E[2].y, E[3].x}, ij{E[4].x, E[3].y};
        const double tterm = E[5].y;
        double r0;
#pragma unroll
        for (int x = 0; x < 5; x++) {
            tb[x] = sj == 0 ? fj[x] : tb[x];
            tc[x] = sk == 0 ? fk[x] : tc[x];
        }
        if (DIR > 0) {
            t = {E[6].x, E[6].y, E[7].x, E[4].y, E[5].x, 0.5 * ij.d};
            r0 = E[7].y;
            lu_fwd_combine(rhs, ta, tb, tc, dg, ij, res);
        } else {
            qv[0] = E[6].x; qv[1] = E[6].y; qv[2] = E[7].x; qv[3] = E[7].y; qv[4] = E[8 % kRow0].x;
            const double ri = E[8 % kRow0].y;
            t = {qv[1] * ri, qv[2] * ri, qv[3] * ri, E[4].y, E[5].x, 0.5 * ij.d};
            r0 = E[9 % kRow0].x;
            lu_bwd_combine(rhs, ta, tb, tc, dg, ij, res);
        }
        const double dp = lu_dp(t, gamma, res);
        lu_product(t, {R[4].x, R[4].y, R[5].x, R[5].y, R[6].y}, dp, res, pc);
#pragma unroll
        for (int x = 0; x < 5; x++) tc[x] = lane_from(behind_k, pc[x]);
        lu_product(t, {R[2].x, R[2].y, R[3].x, R[3].y, R[6].x}, dp, res, pb);
#pragma unroll
        for (int x = 0; x < 5; x++) tb[x] = lane_behind_j<DIR>(pb[x]);
        wait_face(min(s + 1, last));
        load_face(s + 1);
        load_rows(s + 1, NR);
        lds_post(&L.done, s + 1);
        lu_product(t, {R[0].x, R[0].y, R[1].x, R[1].y, r0}, dp, res, ta);
        // face lanes: slot pos + sk = s - (kTile - 1), and the same on the k side
        if (k_out && on) {
#pragma unroll
            for (int x = 0; x < 5; x++) xstore(ko + x * kTile, pc[x]);
        }
        if (j_out && on) {
#pragma unroll
            for (int x = 0; x < 5; x++) xstore(jo + x * kTile, pb[x]);
        }
        jo += kTile * 5;
        ko += kTile * 5;
        if (on) {
            if (fuse_add) {
                const long n = nat0 + (g.Li - 1 - pos);
#pragma unroll
                for (int x = 0; x < 5; x++) q[x * qN + n] = qv[x] + res[x];
            } else {
                // the backward sweep leaves q + dq, the forward sweep dq*, as
                // whole 16-byte pairs, the first one with the time term
                double r[5];
#pragma unroll
                for (int x = 0; x < 5; x++) r[x] = DIR < 0 ? qv[x] + res[x] : res[x];
                dst[0] = make_double2(tterm, r[0]);
                dst[64] = make_double2(r[1], r[2]);
                dst[2 * 64] = make_double2(r[3], r[4]);
            }
        }
        dst += DIR * (kSlF / 2) * 64;
    };
    wait_ops(0);
    load_state(0, E[0]);
    load_rows(0, R[0]);
    wait_face(0);
    load_face(0);
    for (int s = 0; s < g.nsteps; s += 2) {
        step(s, E[0], R[0], E[1], R[1]);
        if (s + 1 < g.nsteps) step(s + 1, E[1], R[1], E[0], R[0]);
    }
}

template <int DIR>
__device__ inline void pipe_body(const SlGeom &g, int tile, double *__restrict__ sl, double gamma, double *ex, int *err,
                                 PipeLds<DIR> &L, const Ext *e, double *__restrict__ q)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (threadIdx.x < kPipePrep) L.prep[threadIdx.x] = threadIdx.x;
    if (threadIdx.x == 64) L.xready = L.done = L.stop = 0;
    for (int x = threadIdx.x; x < kPipeXRing * 10 * kTile; x += kPipeThreads) (&L.x[0][0][0][0])[x] = 0.0;
    __syncthreads();
    const int bj = tile % g.nbj, bk = tile / g.nbj;
    const bool j_pred = DIR > 0 ? bj > 0 : bj + 1 < g.nbj, k_pred = DIR > 0 ? bk > 0 : bk + 1 < g.nbk;
    const bool j_succ = DIR > 0 ? bj + 1 < g.nbj : bj > 0, k_succ = DIR > 0 ? bk + 1 < g.nbk : bk > 0;
    double *exk = ex + (long)g.ntiles * g.exj_tile;
    if (wave == 0) {
        __builtin_amdgcn_s_setprio(3);
        pipe_solve<DIR>(g, tile, sl, gamma, ex + (long)tile * g.exj_tile, exk + (long)tile * g.exk_tile,
                        j_pred || k_pred, j_succ, k_succ, L, err, e, q);
    } else if (wave <= kPipePrep) {
        pipe_prepare<DIR>(g, tile, wave - 1, sl, gamma, L, err);
    } else if (j_pred || k_pred) {
        const bool k_face = (threadIdx.x & 32) != 0, has = k_face ? k_pred : j_pred;
        const int f = threadIdx.x & 7;
        const bool line_ok = has && (k_face ? bj : bk) * kTile + f < (k_face ? g.Lj : g.Lk);
        double *src = !has ? ex : k_face ? exk + (long)(tile - DIR * g.nbj) * g.exk_tile
                                         : ex + (long)(tile - DIR) * g.exj_tile;
        pipe_fetch<DIR>(g, line_ok, DIR > 0 ? f : kTile - 1 - f, src, L, err);
    }
}

// Tile numbers.  The tiles are handed out in the order in which workgroups
// start (a ticket counter): a tile then only ever waits on tiles whose
// workgroups started before it, so the sweep progresses however the launch
// is dispatched and whatever else the device runs, other contexts' sweeps
// among it.  Where tiles by workgroup number are the faster form (fits; the
// hardware's placement of consecutive workgroups suits the sweep), the
// workgroups first count themselves: when the last one has come, all are
// running and every wait ends whatever the order, so each takes the tile of
// its number; a workgroup that has polled kArrivePolls times without seeing
// that (the device is shared) switches the launch to tickets, if it can do
// so before the last one comes.  The last workgroup to finish resets the
// counters for the next launch.
constexpr int kByTicket = 1 << 30, kArrivePolls = 32;
__device__ inline int tile_ticket(int *ctr, int total, bool fits, int *ticket)
{
    if (threadIdx.x == 0) {
        int here = 0, t = (int)blockIdx.x;
        if (fits) {
            here = __hip_atomic_fetch_add(ctr + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
            for (int n = 0; here < total; n++) {
                if (n < kArrivePolls) {
                    __builtin_amdgcn_s_sleep(1);
                    here = __hip_atomic_load(ctr + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else if (__hip_atomic_compare_exchange_strong(ctr + 2, &here, here | kByTicket, __ATOMIC_RELAXED,
                                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    here |= kByTicket;
                }
            }
        }
        if (here != total) t = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *ticket = t;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*ticket);
}
__device__ inline void tile_done(int *ctr, int total)
{
    if (threadIdx.x == 0 &&
        __hip_atomic_fetch_add(ctr + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == total - 1) {
        for (int x = 0; x < kTileCounters; x++)
            __hip_atomic_store(ctr + x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <int DIR>
__global__ void __launch_bounds__(kPipeThreads, 2) k_lu_pipe(SlGeom g, double *__restrict__ sl, double gamma, double *ex,
                                                             int *err, int *ctr, int fits, Ext e, double *q)
{
    __shared__ PipeLds<DIR> L;
    __shared__ int ticket;
    const int flat = tile_ticket(ctr, g.ntiles, fits, &ticket);
    pipe_body<DIR>(g, DIR > 0 ? flat : g.ntiles - 1 - flat, sl, gamma, ex, err, L, &e, q);
    tile_done(ctr, g.ntiles);
}

// ------------------------------------------------------------ batched tiles
// Every block of a context in one launch per phase.  A table holds one
// entry per block (ranges, tiling, operand fields, its part of the
// workspace) and the launch's flat tile numbers run over the blocks one
// after another, tile0 being a block's first.  Fields are offsets from the
// base of the blocks' arena and workspace parts offsets from the
// workspace's bases, all passed as kernel arguments: pointers derived from
// kernel arguments are known to be global memory, so the accesses compile
// to global loads and stores (a pointer read from a table would compile to
// flat ones, which the LDS barriers of the sweep would also wait for).
struct LuBatchEnt {
    Ext e;
    SlGeom g;
    long q, dxidx, inv_j, csnd, dt, rhs;
    long sl, ex;
    int tile0, blk;  // first tile number, block of the context
};

__global__ void __launch_bounds__(kLanes) k_sl_gather_batch(const LuBatchEnt *__restrict__ ents,
                                                        const int *__restrict__ tile_ent, double *arena,
                                                        const double *cfl, int cfl_stride, double *slb, int fp0,
                                                        int parts)
{
    __shared__ double buf[2 * kSlCt * kLanes];
    const int flat = (int)blockIdx.x;
    const LuBatchEnt &b = ents[tile_ent[flat]];
    const Ext e = b.e;
    const SlGeom g = b.g;
    sl_gather_tile(e, g, flat - b.tile0, arena + b.q, arena + b.dxidx, arena + b.inv_j, arena + b.csnd,
                   arena + b.dt, cfl + (long)b.blk * cfl_stride, arena + b.rhs, slb + b.sl,
                   fp0 + (int)blockIdx.y / parts, (int)blockIdx.y % parts, parts, buf);
}

__global__ void __launch_bounds__(kLanes) k_sl_add_batch(const LuBatchEnt *__restrict__ ents,
                                                     const int *__restrict__ tile_ent, double *arena,
                                                     const double *slb, int parts)
{
    __shared__ double buf[2 * kSlCt * kLanes];
    const int flat = (int)blockIdx.x;
    const LuBatchEnt &b = ents[tile_ent[flat]];
    const Ext e = b.e;
    const SlGeom g = b.g;
    sl_add_tile(e, g, flat - b.tile0, slb + b.sl, arena + b.q, kSlOut / 2 + (int)blockIdx.y / parts,
                (int)blockIdx.y % parts, parts, buf);
}

template <int DIR>
__global__ void __launch_bounds__(kPipeThreads, 2) k_lu_pipe_batch(const LuBatchEnt *__restrict__ ents,
                                                                   const int *__restrict__ tile_ent, int total,
                                                                   int fits, double *slb, double *exb,
                                                                   double gamma, int *err, int *ctr, double *arena,
                                                                   int fuse_add)
{
    __shared__ PipeLds<DIR> L;
    __shared__ int ticket;
    const int flat = tile_ticket(ctr, total, fits, &ticket);
    const LuBatchEnt &b = ents[tile_ent[flat]];
    const SlGeom g = b.g;
    const int local = flat - b.tile0;
    const Ext e = b.e;
    pipe_body<DIR>(g, DIR > 0 ? local : g.ntiles - 1 - local, slb + b.sl, gamma, exb + b.ex, err, L, &e,
                   fuse_add ? arena + b.q : nullptr);
    tile_done(ctr, total);
}

// ------------------------------------------------ scalar sweeps (SA model)
// The LU-SGS of the SA working variable (sub_tur_sa.f90:755-812) has the
// same dependencies with one unknown per node:
//   forward   dn* = (rhs + a+ dn*_i-1 + b+ dn*_j-1 + c+ dn*_k-1) / diag
//   backward  dn  = dn* - (a- dn_i+1 + b- dn_j+1 + c- dn_k+1) / diag
// with the node's own a+- = (a +- |a|)/2 (a, b, c the contravariant
// velocities), so a neighbour only supplies its value.  Same tiles and
// skewed clock as the flow sweep; the operands (a, b, c, diag and rhs or
// dn*) are read in place, one i-line per lane (a cache line serves 16
// consecutive steps), and one value per exchange slot crosses a tile edge.
struct SaGeom {
    int nbj, nbk, ntiles, nsteps, Li, Lj, Lk;
    long exj_tile, exk_tile;  // doubles per tile of the j / k exchange regions
};

static SaGeom sa_geom(const Ext &e)
{
    const SlGeom s = sl_geom(e);
    SaGeom g;
    g.nbj = s.nbj;
    g.nbk = s.nbk;
    g.ntiles = s.ntiles;
    g.nsteps = s.nsteps;
    g.Li = s.Li;
    g.Lj = s.Lj;
    g.Lk = s.Lk;
    g.exj_tile = g.exk_tile = (long)(g.Li + kTile - 1) * kTile;
    return g;
}

// a node's new value from the neighbours' (every product and sum rounded by
// itself, as the published sweep's results have them)
template <int DIR>
__device__ inline double sa_node(const double *op, double vi, double vj, double vk)
{
#pragma clang fp contract(off)
    const LuDivisor dg = lu_divisor(op[3]);
    const double a = DIR > 0 ? fabs(op[0]) : -fabs(op[0]), b = DIR > 0 ? fabs(op[1]) : -fabs(op[1]),
                 c = DIR > 0 ? fabs(op[2]) : -fabs(op[2]);
    const double ta = 0.5 * (op[0] + a) * vi, tb = 0.5 * (op[1] + b) * vj, tc = 0.5 * (op[2] + c) * vk;
    const double t = ta + tb + tc;
    return DIR > 0 ? lu_over(op[4] + t, dg) : op[4] - lu_over(t, dg);
}

// The scalar sweep of one tile by one wavefront.  IO gives the operands a,
// b, c, diag and rhs / dn* of a step and takes its result.
//
// What bounds it: the steps in a row (Li + Lj + Lk of them from corner to
// corner of a block, a hop through memory at every tile edge).  A step used
// to take 0.64 us, its operands' latency, as they were read one step ahead
// and the lanes met through LDS; now they are read kSaAhead steps ahead,
// the exchange slots kSaSlotAhead (a slot read earlier than the neighbour
// writes it is polled for), values pass to the next lanes by DPP (j) and
// ds_bpermute (k), and the one division is a product and two fused
// operations on the chain (the quotient is the same).  Forward / backward
// sweep, 12 blocks of 3.2 M nodes in all: 206 / 182 us before, 173 / 154
// now; 24 blocks of 8 M nodes 234 / 203, now 216 / 186.  Steps and slots
// ahead, the 12 blocks: 4, 2 182 / 156; 4, 4 176 / 160; 6, 6 185 / 170; 8, 4
// 175 / 160.
constexpr int kSaOps = 5;  // a, b, c, diag, rhs / dn*
constexpr int kSaAhead = 6, kSaSlotAhead = 3;
template <int DIR, class IO>
__device__ inline void sa_sweep_body(const SaGeom &g, int tile, const IO &io, double *ex, int *err)
{
    const int bj = tile % g.nbj, bk = tile / g.nbj;
    const int l = threadIdx.x, tj = l % kTile, tk = l / kTile;
    const int lj = bj * kTile + tj, lk = bk * kTile + tk;
    const bool active = lj < g.Lj && lk < g.Lk;
    const int sj = DIR > 0 ? tj : kTile - 1 - tj, sk = DIR > 0 ? tk : kTile - 1 - tk;
    const bool j_ring = DIR > 0 ? lj == 0 : lj + 1 >= g.Lj;
    const bool k_ring = DIR > 0 ? lk == 0 : lk + 1 >= g.Lk;
    const bool j_in = active && !j_ring && sj == 0, k_in = active && !k_ring && sk == 0;
    const bool j_out = active && sj == kTile - 1 && (DIR > 0 ? bj + 1 < g.nbj : bj > 0);
    const bool k_out = active && sk == kTile - 1 && (DIR > 0 ? bk + 1 < g.nbk : bk > 0);
    double *exj = ex, *exk = ex + (long)g.ntiles * g.exj_tile;
    // every lane of a tile with a neighbour on that side loads the face
    // lanes' slot run of the step (one contiguous run per load); only the
    // face lanes use it
    const bool j_pred = DIR > 0 ? bj > 0 : bj + 1 < g.nbj;
    const bool k_pred = DIR > 0 ? bk > 0 : bk + 1 < g.nbk;
    double *jin = j_pred ? exj + (long)(DIR > 0 ? tile - 1 : tile + 1) * g.exj_tile + tk : ex;
    double *kin = k_pred ? exk + (long)(DIR > 0 ? tile - g.nbj : tile + g.nbj) * g.exk_tile + tj : ex;
    double *jout = exj + (long)tile * g.exj_tile + tk;
    double *kout = exk + (long)tile * g.exk_tile + tj;
    const int x_last = g.Li + kTile - 2;
    const int behind_k = 4 * (l - DIR * kTile);
    bool failed = false;
    double vi = 0.0;
    auto fetch_slots = [&](int s, unsigned long long &xj, unsigned long long &xk) {
        const long d = (long)min(s, x_last) * kTile;
        xj = xload_bits(jin + (j_pred ? d : 0));
        xk = xload_bits(kin + (k_pred ? d : 0));
    };
    auto step = [&](int s, const double *op, unsigned long long xj, unsigned long long xk) {
        const int pos = s - sj - sk;
        const bool on = active && pos >= 0 && pos < g.Li;
        const bool take_j = on && j_in, take_k = on && k_in;
        bool wait_j = take_j && xj == kSentinel, wait_k = take_k && xk == kSentinel;
        if (__builtin_amdgcn_ballot_w64(wait_j || wait_k)) {
            for (long spins = 0; !failed; spins++) {
                if (wait_j) xj = xload_bits(jin + (long)s * kTile);
                if (wait_k) xk = xload_bits(kin + (long)s * kTile);
                wait_j = wait_j && xj == kSentinel;
                wait_k = wait_k && xk == kSentinel;
                if (!__builtin_amdgcn_ballot_w64(wait_j || wait_k)) break;
                if ((spins & 1023) == 1023 &&
                    (spins > (1L << 21) || __builtin_amdgcn_readfirstlane(__hip_atomic_load(
                                               err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))) {
                    if (l == 0) atomicOr(err, 1);
                    failed = true;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (wait_j) xj = 0;
            if (wait_k) xk = 0;
        }
        if (take_j) xstore_bits(jin + (long)s * kTile, kSentinel);
        if (take_k) xstore_bits(kin + (long)s * kTile, kSentinel);
        const double nj = lane_behind_j<DIR>(vi), nk = lane_from(behind_k, vi);
        const double vj = j_ring ? 0.0 : j_in ? __longlong_as_double((long long)xj) : nj;
        const double vk = k_ring ? 0.0 : k_in ? __longlong_as_double((long long)xk) : nk;
        const double res = sa_node<DIR>(op, vi, vj, vk);
        vi = on ? res : 0.0;
        if (on) {
            io.store(s, pos, res);
            if (j_out) xstore(jout + (long)(pos + sk) * kTile, res);
            if (k_out) xstore(kout + (long)(pos + sj) * kTile, res);
        }
    };
    double op[kSaAhead][kSaOps];
    unsigned long long xj[kSaAhead], xk[kSaAhead];
#pragma unroll
    for (int u = 0; u < kSaAhead; u++) io.load(u, u - sj - sk, op[u]);
#pragma unroll
    for (int u = 0; u < kSaSlotAhead; u++) fetch_slots(u, xj[u], xk[u]);
    // (steps past the last find every lane off)
    for (int s = 0; s < g.nsteps; s += kSaAhead) {
#pragma unroll
        for (int u = 0; u < kSaAhead; u++) {
            constexpr int A = kSaAhead;
            fetch_slots(s + u + kSaSlotAhead, xj[(u + kSaSlotAhead) % A], xk[(u + kSaSlotAhead) % A]);
            step(s + u, op[u], xj[u], xk[u]);
            io.load(s + u + A, s + u + A - sj - sk, op[u]);
        }
    }
}

// operands and results in place, one i-line of a block per lane: cu = a, b,
// c, diag (component stride N); forward reads rhs and writes dns, backward
// reads dns and writes dn
template <int DIR>
struct SaInPlace {
    const double *cu, *src;
    double *out;
    long N, n0;  // n0: the lane's first node in storage (a valid one on inactive lanes)
    int Li;
    __device__ SaInPlace(const Ext &e, const SaGeom &g, int tile, const double *c, const double *rhs, double *dns,
                         double *dn)
        : cu(c), src(DIR > 0 ? rhs : dns), out(DIR > 0 ? dns : dn), N(e.n), Li(g.Li)
    {
        const int l = threadIdx.x;
        n0 = e.ix(e.is1, e.js1 + min(tile % g.nbj * kTile + l % kTile, g.Lj - 1),
                  e.ks1 + min(tile / g.nbj * kTile + l / kTile, g.Lk - 1));
    }
    __device__ long node(int pos) const { return n0 + (DIR > 0 ? pos : Li - 1 - pos); }
    __device__ void load(int, int pos, double *op) const
    {
        const long n = node(min(max(pos, 0), Li - 1));
#pragma unroll
        for (int f = 0; f < 4; f++) op[f] = cu[f * N + n];
        op[4] = src[n];
    }
    __device__ void store(int, int pos, double v) const { out[node(pos)] = v; }
};

template <int DIR>
__global__ void __launch_bounds__(kLanes) k_sa_tiles(Ext e, SaGeom g, const double *__restrict__ cu,
                                                      const double *__restrict__ rhs, double *__restrict__ dns,
                                                      double *__restrict__ dn, double *ex, int *err, int *ctr)
{
    __shared__ int ticket;
    const int flat = tile_ticket(ctr, g.ntiles, false, &ticket);
    const int tile = DIR > 0 ? flat : g.ntiles - 1 - flat;
    sa_sweep_body<DIR>(g, tile, SaInPlace<DIR>(e, g, tile, cu, rhs, dns, dn), ex, err);
    tile_done(ctr, g.ntiles);
}

struct SaBatchEnt {
    Ext e;
    SaGeom g;
    long cu, rhs, dns, dn, ex;
    long sl;  // the block's part of the SA sweep layout (offset from its base)
    long nut;
    int tile0;
};

template <int DIR>
__global__ void __launch_bounds__(kLanes) k_sa_tiles_batch(const SaBatchEnt *__restrict__ ents,
                                                            const int *__restrict__ tile_ent, int total,
                                                            double *arena, double *exb, int *err,
                                                            int *ctr)
{
    __shared__ int ticket;
    const int flat = tile_ticket(ctr, total, false, &ticket);
    const SaBatchEnt &b = ents[tile_ent[flat]];
    const Ext e = b.e;
    const SaGeom g = b.g;
    const int local = flat - b.tile0, tile = DIR > 0 ? local : g.ntiles - 1 - local;
    sa_sweep_body<DIR>(g, tile,
                       SaInPlace<DIR>(e, g, tile, arena + b.cu, arena + b.rhs, arena + b.dns, arena + b.dn),
                       exb + b.ex, err);
    tile_done(ctr, total);
}

// ---- scalar sweeps over an SA sweep layout (every block in one launch)
// The operands a, b, c, diag and the right-hand side of every computed node
// are moved into a sweep layout ordered (tile, step, operand, lane): at
// step t, lane l of a tile reads its five operands as five rows of TT
// consecutive doubles, whole lines for the wavefront, where the natural
// layout has each lane on a line of its own.  Row t of lane (tj, tk) holds
// the node li = t - tj - tk of the lane's i-line; the backward sweep's step
// s reads row nsteps-1-s for every lane (its skewed clock runs the same
// rows in reverse).  The forward sweep leaves dnut* in the rhs operand's
// slot and the backward sweep dnut there; a last pass adds it to nut.
__host__ __device__ inline long sa_slot(const SaGeom &g, int tile, int t, int f, int l)
{
    return (((long)tile * g.nsteps + t) * kSaOps + f) * kLanes + l;
}

// node of (tile, line, li) of a block and whether the line exists
__device__ inline long sa_nat(const Ext &e, const SaGeom &g, int tile, int line, int li)
{
    const int tj = line % kTile, tk = line / kTile;
    return e.ix(e.is1 + li, e.js1 + (tile % g.nbj) * kTile + tj, e.ks1 + (tile / g.nbj) * kTile + tk);
}
__device__ inline bool sa_line_ok(const SaGeom &g, int tile, int line)
{
    return (tile % g.nbj) * kTile + line % kTile < g.Lj && (tile / g.nbj) * kTile + line / kTile < g.Lk;
}

// Natural layout <-> SA sweep layout for one tile (one workgroup of TT
// threads), the walk of the flow sweep's layout passes: chunks of CT steps,
// a natural-side thread handling CT consecutive nodes of a line, an
// XOR-swizzled [CT][TT] LDS buffer in between.  TO_SL: cu (4 operands,
// component stride N) and rhs into the layout; otherwise nut += the layout's
// last operand.
template <bool TO_SL>
__device__ inline void sa_layout_tile(const Ext &e, const SaGeom &g, int tile, const double *__restrict__ cu,
                                      const double *__restrict__ rhs, double *__restrict__ nut, double *__restrict__ L,
                                      int f, int part, int parts, double *buf /* [CT][TT] */)
{
    constexpr int CT = TO_SL ? kSlCt : kSaRetCt, TT = kLanes, lstep = TT / CT;
    const int x = threadIdx.x;
    const int ii_n = x % CT;
    const int tj = x % kTile, tk = x / kTile;
    const bool me_ok = sa_line_ok(g, tile, x);
    const long N = e.n;
    const SlChunks ch(g.nsteps, CT, part, parts);
    for (int t0 = ch.t0; t0 < ch.t1; t0 += CT) {
        int nat[CT];  // node offsets fit 32 bits (blocks below 2^31 nodes)
#pragma unroll
        for (int m = 0; m < CT; m++) {
            const int line = m * lstep + x / CT;
            const int li = t0 + ii_n - line % kTile - line / kTile;
            nat[m] = (t0 + ii_n < g.nsteps && li >= 0 && li < g.Li && sa_line_ok(g, tile, line))
                         ? (int)sa_nat(e, g, tile, line, li) : -1;
        }
        if (TO_SL) {
            const double *src = f < 4 ? cu + f * N : rhs;
            double v[CT];
#pragma unroll
            for (int m = 0; m < CT; m++) v[m] = nat[m] >= 0 ? src[nat[m]] : 0.0;
#pragma unroll
            for (int m = 0; m < CT; m++) {
                const int line = m * lstep + x / CT;
                buf[ii_n * TT + (line ^ ii_n)] = v[m];
            }
            __syncthreads();
            if (me_ok) {
#pragma unroll
                for (int ii = 0; ii < CT; ii++) {
                    const int t = t0 + ii, li = t - tj - tk;
                    if (t < g.nsteps && li >= 0 && li < g.Li) L[sa_slot(g, tile, t, f, x)] = buf[ii * TT + (x ^ ii)];
                }
            }
            __syncthreads();
        } else {
            if (me_ok) {
#pragma unroll
                for (int ii = 0; ii < CT; ii++) {
                    const int t = t0 + ii, li = t - tj - tk;
                    buf[ii * TT + (x ^ ii)] =
                        (t < g.nsteps && li >= 0 && li < g.Li) ? L[sa_slot(g, tile, t, kSaOps - 1, x)] : 0.0;
                }
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < CT; m++) {
                const int line = m * lstep + x / CT;
                if (nat[m] >= 0) nut[nat[m]] = nut[nat[m]] + buf[ii_n * TT + (line ^ ii_n)];
            }
            __syncthreads();
        }
    }
}

template <bool TO_SL>
__global__ void __launch_bounds__(kLanes) k_sa_layout_batch(const SaBatchEnt *__restrict__ ents,
                                                        const int *__restrict__ tile_ent, double *arena,
                                                        double *slbase, int parts)
{
    __shared__ double buf[(TO_SL ? kSlCt : kSaRetCt) * kLanes];
    const int flat = (int)xcd_slab(blockIdx.x, gridDim.x);
    const SaBatchEnt &b = ents[tile_ent[flat]];
    const Ext e = b.e;
    const SaGeom g = b.g;
    sa_layout_tile<TO_SL>(e, g, flat - b.tile0, arena + b.cu, arena + b.rhs, arena + b.nut, slbase + b.sl,
                          (int)blockIdx.y / parts, (int)blockIdx.y % parts, parts, buf);
}

// operands and results in the SA sweep layout; rows: the tile's row 0 at
// this lane
template <int DIR>
struct SaRows {
    double *rows;
    int nsteps;
    __device__ double *row(int s) const
    {
        const int sc = min(s, nsteps - 1);
        return rows + (long)(DIR > 0 ? sc : nsteps - 1 - sc) * kSaOps * kLanes;
    }
    __device__ void load(int s, int, double *op) const
    {
        const double *p = row(s);
#pragma unroll
        for (int f = 0; f < kSaOps; f++) op[f] = p[f * kLanes];
    }
    __device__ void store(int s, int, double v) const { row(s)[(kSaOps - 1) * kLanes] = v; }
};

template <int DIR>
__global__ void __launch_bounds__(kLanes) k_sa_sl_batch(const SaBatchEnt *__restrict__ ents,
                                                         const int *__restrict__ tile_ent, int total,
                                                         double *slbase, double *exb, int *err, int *ctr)
{
    __shared__ int ticket;
    const int flat = tile_ticket(ctr, total, false, &ticket);
    const SaBatchEnt &b = ents[tile_ent[flat]];
    const SaGeom g = b.g;
    const int local = flat - b.tile0, tile = DIR > 0 ? local : g.ntiles - 1 - local;
    sa_sweep_body<DIR>(g, tile, SaRows<DIR>{slbase + b.sl + sa_slot(g, tile, 0, 0, (int)threadIdx.x), g.nsteps},
                       exb + b.ex, err);
    tile_done(ctr, total);
}

static long lusgs_tiles(const Ext &e)
{
    const SlGeom g = sl_geom(e);
    return g.Li > 0 && g.Lj > 0 && g.Lk > 0 ? g.ntiles : 0;
}

void lusgs_ws_sizes(const Ext &e, long *sl_n, long *ex_n)
{
    const SlGeom g = sl_geom(e);
    const bool any = lusgs_tiles(e) > 0;
    *sl_n = any ? (long)g.ntiles * g.nsteps * kSlF * kLanes : 0;
    *ex_n = any ? (long)g.ntiles * (g.exj_tile + g.exk_tile) : 0;
}

// Whether the backward sweep adds dq to q itself (and the add pass is
// skipped).  Its stores then go to the natural layout, one line per lane.
// On one block's launch that is the faster form up to about a million
// computed nodes (step of 33^3 0.256 against 0.264 ms, 65^3 0.531 / 0.537,
// 97^3 0.892 / 0.896) and dearer on larger ones (129^3 1.576 / 1.560).  In
// the batched sweeps it costs more than the pass it saves (12 blocks of 3.2
// M nodes: +0.25 ms against 0.10 ms), so batched launches never fuse.
// ACFD_LU_FUSED_ADD=0/1 forces either form.
constexpr long kFuseAddMaxNodes = 1L << 20;
static bool fused_add(long launch_nodes, bool batched = false)
{
    const char *v = std::getenv("ACFD_LU_FUSED_ADD");
    if (v) return std::atoi(v) != 0;
    return !batched && launch_nodes < kFuseAddMaxNodes;
}
static long computed_nodes(const Ext &e)
{
    return (long)(e.ie1 - e.is1 + 1) * (e.je1 - e.js1 + 1) * (e.ke1 - e.ks1 + 1);
}

static long round_up32(long n) { return (n + 31) / 32 * 32; }
static void batch_residency(LuBatch *b);

// blocks of the batch in launch order: longest sweep first
static std::vector<int> batch_order(int nblk, const Ext *e)
{
    std::vector<int> order;
    for (int m = 0; m < nblk; m++)
        if (lusgs_tiles(e[m]) > 0) order.push_back(m);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        const SlGeom ga = sl_geom(e[a]), gb = sl_geom(e[b]);
        return ga.nsteps + ga.nbj + ga.nbk > gb.nsteps + gb.nbj + gb.nbk;
    });
    return order;
}

void lusgs_batch_ws(int nblk, const Ext *e, long *sl_n, long *ex_n)
{
    long a = 0, b = 0;
    for (int m : batch_order(nblk, e)) {
        const SlGeom g = sl_geom(e[m]);
        a += round_up32((long)g.ntiles * g.nsteps * kSlF * kLanes);
        b += round_up32((long)g.ntiles * (g.exj_tile + g.exk_tile));
    }
    *sl_n = a;
    *ex_n = b;
}

int lusgs_batch_make(int nblk, const Ext *e, const Fields *f, double *arena, double *sl, double *ex,
                     LuBatch *out)
{
    std::vector<LuBatchEnt> ents;
    std::vector<int> te;
    long so = 0, xo = 0;
    for (int m : batch_order(nblk, e)) {
        const SlGeom g = sl_geom(e[m]);
        LuBatchEnt b;
        b.e = e[m];
        b.g = g;
        b.q = f[m].q - arena;
        b.dxidx = f[m].dxidx - arena;
        b.inv_j = f[m].inv_j - arena;
        b.csnd = f[m].pri + 6 * e[m].n - arena;
        b.dt = f[m].dt - arena;
        b.blk = m;
        b.rhs = f[m].rhs - arena;
        b.sl = so;
        b.ex = xo;
        b.tile0 = (int)te.size();
        so += round_up32((long)g.ntiles * g.nsteps * kSlF * kLanes);
        xo += round_up32((long)g.ntiles * (g.exj_tile + g.exk_tile));
        for (int t = 0; t < g.ntiles; t++) te.push_back((int)ents.size());
        ents.push_back(b);
    }
    out->arena = arena;
    out->sl = sl;
    out->ex = ex;
    out->nent = (int)ents.size();
    out->total = (int)te.size();
    for (const LuBatchEnt &b : ents) out->nsteps = std::max(out->nsteps, b.g.nsteps);
    if (ents.empty()) return 0;
    batch_residency(out);
    long total = 0;
    for (const LuBatchEnt &b : ents) total += computed_nodes(b.e);
    out->fuse_add = fused_add(total, true) ? 1 : 0;
    if (hipMalloc(&out->ents, ents.size() * sizeof(LuBatchEnt)) != hipSuccess) return 1;
    if (hipMalloc((void **)&out->tile_ent, te.size() * sizeof(int)) != hipSuccess) return 1;
    if (hipMemcpy(out->ents, ents.data(), ents.size() * sizeof(LuBatchEnt), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(out->tile_ent, te.data(), te.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
        return 1;
    return 0;
}

void lusgs_batch_free(LuBatch *b)
{
    if (b->ents) (void)hipFree(b->ents);
    if (b->tile_ent) (void)hipFree(b->tile_ent);
    b->ents = nullptr;
    b->tile_ent = nullptr;
    b->nent = b->total = 0;
}

// workgroups of the kernel that the device holds (0: unknown)
template <typename K>
static int resident_wgs(K kernel, int threads)
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess)
        return 0;
    return cus * per_cu;
}

// ACFD_LU_TICKETS=1: by ticket whatever fits
static bool tickets_only()
{
    const char *t = std::getenv("ACFD_LU_TICKETS");
    return t && std::atoi(t) == 1;
}

void lusgs_resident(int *wgs)
{
    const bool t = tickets_only();
    wgs[0] = t ? 0 : resident_wgs(k_lu_pipe<1>, kPipeThreads);
    wgs[1] = t ? 0 : resident_wgs(k_lu_pipe<-1>, kPipeThreads);
}

// Whether a sweep of `tiles` tiles tries to run them by workgroup number (see
// tile_ticket).  Forward / backward sweep, us, by ticket, by number after
// counting and by number at once: 97^3 (169 tiles) 255 / 274, -, 254 / 273;
// 129^3 (256) 391 / 382, 360 / 359, 358 / 356; 161^3 (400) 584 / 548, 550 /
// 532, 538 / 519.  Fewer tiles gain nothing by it.  The SA model's sweeps
// are at least as fast by ticket (both of two blocks of 1.2 M nodes 595 ->
// 581 us with the passes around them) and always go that way.
constexpr int kFitsMin = 192;
static bool tile_fits(int tiles, int resident) { return tiles >= kFitsMin && tiles <= resident; }

static void batch_residency(LuBatch *b)
{
    if (tickets_only()) return;
    b->fits[0] = tile_fits(b->total, resident_wgs(k_lu_pipe_batch<1>, kPipeThreads));
    b->fits[1] = tile_fits(b->total, resident_wgs(k_lu_pipe_batch<-1>, kPipeThreads));
}

template <int DIR>
static void launch_pipe_batch(hipStream_t s, const LuBatch &b, double gamma, int *err, int *ctr)
{
    hipLaunchKernelGGL((k_lu_pipe_batch<DIR>), dim3((unsigned)b.total), dim3(kPipeThreads), 0, s,
                       (const LuBatchEnt *)b.ents, b.tile_ent, b.total, b.fits[DIR > 0 ? 0 : 1], b.sl, b.ex, gamma,
                       err, ctr, b.arena, DIR < 0 && b.fuse_add ? 1 : 0);
}

// Phases 1-4 of the LU-SGS update for every block of the batch at once
// (phase 0, the per-node preparation, stays per block).  geo_cached: the
// sweep layout already holds this batch's grid operands (phase 1 then
// gathers the other fields only).
int launch_lusgs_batch(hipStream_t s, const LuBatch &b, int phase, double gamma, int *err, int *ctr, const double *cfl,
                       int cfl_stride, int geo_cached)
{
    if (b.total <= 0 || phase < 1 || phase > 4) return 0;
    const LuBatchEnt *ents = (const LuBatchEnt *)b.ents;
    const int fp0 = geo_cached ? kSlGeoPairs : 0, pairs = phase == 1 ? kSlF / 2 - fp0 : kSlF / 2 - kSlOut / 2;
    const int parts = sl_parts(b.total, pairs, b.nsteps, kSlCt);
    if (phase == 1)
        hipLaunchKernelGGL(k_sl_gather_batch, dim3((unsigned)b.total, (unsigned)(pairs * parts)), dim3(kLanes), 0, s, ents,
                           b.tile_ent, b.arena, cfl, cfl_stride, b.sl, fp0, parts);
    else if (phase == 2) launch_pipe_batch<1>(s, b, gamma, err, ctr);
    else if (phase == 3) launch_pipe_batch<-1>(s, b, gamma, err, ctr);
    else if (!b.fuse_add)
        hipLaunchKernelGGL(k_sl_add_batch, dim3((unsigned)b.total, (unsigned)(pairs * parts)), dim3(kLanes), 0, s, ents,
                           b.tile_ent, b.arena, (const double *)b.sl, parts);
    ACFD_CHECK_LAUNCH();
    return 0;
}

// ---- scalar sweeps: host side
// both SA sweeps of one block (ex: sentinel-filled, at least
// ntiles * (exj_tile + exk_tile) doubles -- less than the flow sweep's)
int launch_sa_sweeps(hipStream_t s, const Ext &e, const double *cu, const double *rhs, double *dns,
                     double *dn, double *ex, int *err, int *ctr)
{
    const SaGeom g = sa_geom(e);
    if (g.Li <= 0 || g.Lj <= 0 || g.Lk <= 0) return 0;
    hipLaunchKernelGGL((k_sa_tiles<1>), dim3((unsigned)g.ntiles), dim3(kLanes), 0, s, e, g, cu, rhs, dns, dn, ex, err,
                       ctr);
    hipLaunchKernelGGL((k_sa_tiles<-1>), dim3((unsigned)g.ntiles), dim3(kLanes), 0, s, e, g, cu, rhs, dns, dn, ex, err,
                       ctr);
    ACFD_CHECK_LAUNCH();
    return 0;
}

void sa_batch_sl(int nblk, const Ext *e, long *sl_n)
{
    long so = 0;
    for (int m = 0; m < nblk; m++) {
        const SaGeom g = sa_geom(e[m]);
        if (g.Li <= 0 || g.Lj <= 0 || g.Lk <= 0) continue;
        so += round_up32((long)g.ntiles * g.nsteps * kSaOps * kLanes);
    }
    *sl_n = so;
}

int sa_batch_make(int nblk, const Ext *e, const Fields *f, double *arena, double *ex, double *sl,
                  LuBatch *out)
{
    std::vector<SaBatchEnt> ents;
    std::vector<int> te;
    long xo = 0, so = 0;
    for (int m : batch_order(nblk, e)) {
        const SaGeom g = sa_geom(e[m]);
        if (!f[m].w_sa) continue;
        SaBatchEnt b;
        b.e = e[m];
        b.g = g;
        b.cu = f[m].w_dqs - arena;
        b.rhs = f[m].sa_rhs - arena;
        b.dns = f[m].w_sa + 8 * e[m].n - arena;
        b.dn = f[m].w_dq - arena;
        b.nut = f[m].nut - arena;
        b.ex = xo;
        b.sl = so;
        b.tile0 = (int)te.size();
        xo += round_up32((long)g.ntiles * (g.exj_tile + g.exk_tile));
        so += round_up32((long)g.ntiles * g.nsteps * kSaOps * kLanes);
        for (int t = 0; t < g.ntiles; t++) te.push_back((int)ents.size());
        ents.push_back(b);
    }
    out->arena = arena;
    out->ex = ex;
    out->sl = sl;
    out->nent = (int)ents.size();
    out->total = (int)te.size();
    for (const SaBatchEnt &b : ents) out->nsteps = std::max(out->nsteps, b.g.nsteps);
    if (ents.empty()) return 0;
    if (hipMalloc(&out->ents, ents.size() * sizeof(SaBatchEnt)) != hipSuccess) return 1;
    if (hipMalloc((void **)&out->tile_ent, te.size() * sizeof(int)) != hipSuccess) return 1;
    if (hipMemcpy(out->ents, ents.data(), ents.size() * sizeof(SaBatchEnt), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(out->tile_ent, te.data(), te.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
        return 1;
    return 0;
}

// SA sweeps over the SA sweep layout: phase 0 moves a, b, c, diag and rhs
// into the layout, 1 / -1 run the forward / backward sweep, 2 adds dnut
// to nut
int launch_sa_sl_batch(hipStream_t s, const LuBatch &b, int *err, int *ctr, int phase)
{
    if (b.total <= 0 || !b.sl) return 0;
    const SaBatchEnt *ents = (const SaBatchEnt *)b.ents;
    const dim3 gr((unsigned)b.total);
    const int fields = phase == 0 ? kSaOps : 1, parts = sl_parts(b.total, fields, b.nsteps, phase == 0 ? kSlCt : kSaRetCt);
    const dim3 gl((unsigned)b.total, (unsigned)(fields * parts));
    if (phase == 0)
        hipLaunchKernelGGL((k_sa_layout_batch<true>), gl, dim3(kLanes), 0, s, ents, b.tile_ent, b.arena, b.sl, parts);
    else if (phase == 2)
        hipLaunchKernelGGL((k_sa_layout_batch<false>), gl, dim3(kLanes), 0, s, ents, b.tile_ent, b.arena, b.sl, parts);
    else if (phase == 1)
        hipLaunchKernelGGL((k_sa_sl_batch<1>), gr, dim3(kLanes), 0, s, ents, b.tile_ent, b.total, b.sl,
                           b.ex, err, ctr);
    else
        hipLaunchKernelGGL((k_sa_sl_batch<-1>), gr, dim3(kLanes), 0, s, ents, b.tile_ent, b.total, b.sl,
                           b.ex, err, ctr);
    ACFD_CHECK_LAUNCH();
    return 0;
}

// the SA sweeps of every block of the batch (dir 0: both, in order)
int launch_sa_batch(hipStream_t s, const LuBatch &b, int *err, int *ctr, int dir)
{
    if (b.total <= 0) return 0;
    const SaBatchEnt *ents = (const SaBatchEnt *)b.ents;
    const dim3 gr((unsigned)b.total);
    if (dir >= 0)
        hipLaunchKernelGGL((k_sa_tiles_batch<1>), gr, dim3(kLanes), 0, s, ents, b.tile_ent, b.total,
                           b.arena, b.ex, err, ctr);
    if (dir <= 0)
        hipLaunchKernelGGL((k_sa_tiles_batch<-1>), gr, dim3(kLanes), 0, s, ents, b.tile_ent, b.total,
                           b.arena, b.ex, err, ctr);
    ACFD_CHECK_LAUNCH();
    return 0;
}

int launch_fill_sentinel(hipStream_t s, double *p, long n)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_fill_sentinel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    ACFD_CHECK_LAUNCH();
    return 0;
}

template <int DIR>
static void launch_pipe(hipStream_t s, const SlGeom &g, const LuWs &ws, double gamma, const Ext &e, double *q)
{
    hipLaunchKernelGGL((k_lu_pipe<DIR>), dim3((unsigned)g.ntiles), dim3(kPipeThreads), 0, s, g, ws.sl, gamma, ws.ex,
                       ws.err, ws.ctr, tile_fits(g.ntiles, ws.resident[DIR > 0 ? 0 : 1]), e, q);
}

// Phases of one LU-SGS update:
//   0 rhs and, for hyperplanes, spectral radii and diag (and dq* and dq
//     cleared),
//   1 tiles: gather the operands, with the time term phi/dt, into the
//     sweep layout (with geo_cached,
//     which says that it already holds this block's grid operands in this
//     tiling, all but those),
//   2 forward sweep, 3 backward sweep,
//   4 q += dq (tiles: from the sweep layout, or fused into the backward
//     sweep, which then stores q + dq itself).
// variant 0 = hyperplanes, 1 = tiles.
int launch_lusgs_phase(hipStream_t s, const Ext &e, const Fields &f, const Consts &c, const double *cfl,
                       int variant, const LuWs *ws, int phase, int geo_cached)
{
    int Li = e.ie1 - e.is1 + 1, Lj = e.je1 - e.js1 + 1, Lk = e.ke1 - e.ks1 + 1;
    const bool tiles = variant == 1 && ws && ws->sl && ws->ex;
    const bool empty = Li <= 0 || Lj <= 0 || Lk <= 0;
    if (phase == 0) {
        hipLaunchKernelGGL(k_lu_prep, lu_prep_grid(e), dim3(64, 4, 1), 0, s, e, f.pri, f.dxidx, f.dt, f.rhsi,
                           f.rhsv, f.rhs, f.w_r, f.w_diag, f.w_dqs, f.w_dq, cfl, tiles ? 1 : 0);
    } else if (empty) {
        return 0;
    } else if (tiles) {
        const SlGeom g = sl_geom(e);
        const bool fuse = fused_add(computed_nodes(e));
        if (phase == 1) launch_layout(s, 0, e, g, f, *ws, cfl, geo_cached ? kSlGeoPairs : 0);
        else if (phase == 2) launch_pipe<1>(s, g, *ws, c.gamma, e, nullptr);
        else if (phase == 3) launch_pipe<-1>(s, g, *ws, c.gamma, e, fuse ? f.q : nullptr);
        else if (!fuse) launch_layout(s, 1, e, g, f, *ws);
    } else if (phase == 4) {
        Box b{e.is1, e.ie1, e.js1, e.je1, e.ks1, e.ke1};
        hipLaunchKernelGGL(k_add5, box_grid(b), dim3(64, 4, 1), 0, s, e, b, f.q, f.w_dq);
    } else if (phase == 2 || phase == 3) {
        LuArgs a{e, f.q, f.dxidx, f.inv_j, f.w_r, f.w_diag, f.rhs, f.w_dqs, f.w_dq, c.gamma};
        const bool fwd = phase == 2;
        int L = Li + Lj + Lk - 2;
        for (int l = 0; l < L; l++) {
            int ja = max(0, l - (Li - 1) - (Lk - 1)), jb = min(Lj - 1, l);
            int ka = max(0, l - (Li - 1) - (Lj - 1)), kb = min(Lk - 1, l);
            dim3 gr((jb - ja + 64) / 64, (kb - ka + 4) / 4, 1);
            if (fwd) hipLaunchKernelGGL((k_lu_plane<1>), gr, dim3(64, 4, 1), 0, s, a, l, ja, ka);
            else hipLaunchKernelGGL((k_lu_plane<-1>), gr, dim3(64, 4, 1), 0, s, a, l, ja, ka);
        }
    }
    ACFD_CHECK_LAUNCH();
    return 0;
}

}  // namespace acfd
