// gfx950 kernels of the viscous residual and the Spalart-Allmaras model.
//
//   visrhs (src/visrhs.f:2-287)        k_visrhs      one workgroup per 32x8 tile of cells:
//                                                    per-cell primitives, coefficients and
//                                                    cross terms once into LDS, then each
//                                                    cell's thin-layer fluxes from there
//   vmu_sa (src/samodel2d.f:2-197)     k_sa_prim     laminar viscosity, u, v (all cells)
//                                      k_turbc       SA boundary conditions (one workgroup per
//                                                    instance); the final ones with the
//                                                    eddy viscosity of the halo ring
//                                      k_sa_rhs      convection, diffusion, source and the
//                                                    two scalar tridiagonal systems: what
//                                                    the stencil reads once per cell of a
//                                                    32x8 tile in LDS, then each cell's row
//                                      k_sa_solve_j  tridiagonal solve along j, one wave per row
//                                      k_sa_solve_k  tridiagonal solve along k, 8 or 16 adjacent
//                                                    j columns per workgroup, nu-tilde update and
//                                                    eddy viscosity
//
// Operand order follows the reference expressions (built with
// -ffp-contract=off), so results agree with the reference to the rounding of
// the device's sqrt/div/pow; the line solves run in parts (part_line,
// part_columns), which changes their rounding only.
#include "ot2d_dev.h"

namespace ot2d {

__device__ __forceinline__ double sqd(double a) { return a * a; }
__device__ __forceinline__ int imx(int a, int b) { return a > b ? a : b; }

// ====================================================================== visrhs
struct VisPrim {
  double u, v, e, vnu, gkap;
};

// per-cell quantities of the visrhs line loops (src/visrhs.f:47-57)
__device__ __forceinline__ VisPrim vis_prim_of(double q1, double q2, double q3, double q4, double turm, double ggm1,
                                               double c2b, double c2bp, double prtr) {
  VisPrim p;
  double ra = 1. / q1;
  p.u = q2 * ra;
  p.v = q3 * ra;
  p.e = q4 * ra - .5 * (sqd(p.u) + sqd(p.v));
  double tt = ggm1 * p.e;
  double vmue = c2bp * tt * sqrt(tt) / (c2b + tt);
  p.vnu = vmue + turm;
  p.gkap = vmue + prtr * turm;
  return p;
}
__device__ __forceinline__ VisPrim vis_prim(const DevMesh& M, long long i, double c2b, double c2bp, double prtr) {
  return vis_prim_of(M.q[0][i], M.q[1][i], M.q[2][i], M.q[3][i], M.turmu[i], M.c.ggm1, c2b, c2bp, prtr);
}

struct VisCoef {
  double c1, c2, c5, c4;          // thin-layer coefficients (b1v.. or a1v..)
  double d1, d2, d4, d5, d7;      // cross-derivative coefficients
};

// metrics of a cell and the reciprocal of its Jacobian q(.,.,nq)
struct VisMet {
  double xx, xy, yx, yy, r;
};
__device__ __forceinline__ VisMet vis_met(const DevMesh& M, long long i) {
  VisMet m;
  m.xx = M.xx[i];
  m.xy = M.xy[i];
  m.yx = M.yx[i];
  m.yy = M.yy[i];
  m.r = 1. / M.q[M.nq - 1][i];
  return m;
}

// coefficients of one line direction at a cell: the thin-layer terms from
// the cell's metric pair (ma, mb) = (yx, yy) along eta, (xx, xy) along xi,
// and the cross terms from its two neighbours m, p across the line
// (src/visrhs.f:59-92 eta, 184-217 xi; both use the same expressions)
__device__ __forceinline__ VisCoef vis_coef(double ma, double mb, double rj, const VisMet& m, const VisMet& p,
                                            const VisPrim& c, double dre, double gkpr) {
  VisCoef o;
  double b4 = (sqd(ma) + sqd(mb)) * rj;
  o.c1 = (b4 + sqd(ma) / 3. * rj) * c.vnu * dre;
  o.c2 = (b4 + sqd(mb) / 3. * rj) * c.vnu * dre;
  o.c5 = (ma * mb / 3. * rj) * c.vnu * dre;
  o.c4 = b4 * gkpr * c.gkap * dre;
  double t;
  t = (4. / 3. * m.xx * m.yx + m.xy * m.yy) * m.r;
  t = t + (4. / 3. * p.xx * p.yx + p.xy * p.yy) * p.r;
  o.d1 = c.vnu * dre * t;
  t = (4. / 3. * m.xy * m.yy + m.xx * m.yx) * m.r;
  t = t + (4. / 3. * p.xy * p.yy + p.xx * p.yx) * p.r;
  o.d2 = c.vnu * dre * t;
  t = (m.xy * m.yy + m.xx * m.yx) * m.r;
  t = t + (p.xy * p.yy + p.xx * p.yx) * p.r;
  o.d4 = t * gkpr * c.gkap * dre;
  t = (-2. / 3. * m.xy * m.yx + m.xx * m.yy) * m.r;
  t = t + (-2. / 3. * p.xy * p.yx + p.xx * p.yy) * p.r;
  o.d5 = c.vnu * dre * t;
  t = (-2. / 3. * m.xx * m.yy + m.xy * m.yx) * m.r;
  t = t + (-2. / 3. * p.xx * p.yy + p.xy * p.yx) * p.r;
  o.d7 = c.vnu * dre * t;
  return o;
}

// eta direction (j = const line) coefficients of cell (j,k) from global memory
__device__ __forceinline__ VisCoef eta_coef(const DevMesh& M, int j, int k, const VisPrim& p, double dre,
                                            double gkpr) {
  long long i = cell(M, j, k);
  return vis_coef(M.yx[i], M.yy[i], 1. / M.q[M.nq - 1][i], vis_met(M, cell(M, j - 1, k)),
                  vis_met(M, cell(M, j + 1, k)), p, dre, gkpr);
}

// xi direction (k = const line) coefficients of cell (j,k) from global memory
__device__ __forceinline__ VisCoef xi_coef(const DevMesh& M, int j, int k, const VisPrim& p, double dre,
                                           double gkpr) {
  long long i = cell(M, j, k);
  return vis_coef(M.xx[i], M.xy[i], 1. / M.q[M.nq - 1][i], vis_met(M, cell(M, j, k - 1)),
                  vis_met(M, cell(M, j, k + 1)), p, dre, gkpr);
}

struct Tri { double f2, f3, f4; };

// thin-layer flux across the face between cells a (low) and b (high) of a line
__device__ __forceinline__ Tri vis_face(const VisPrim& pa, const VisCoef& ca, const VisPrim& pb, const VisCoef& cb) {
  double b1 = cb.c1 + ca.c1, b2 = cb.c2 + ca.c2, b5 = cb.c5 + ca.c5;
  double t4 = pb.u * cb.c1 + pa.u * ca.c1;
  double t5 = pb.v * cb.c2 + pa.v * ca.c2;
  double t6 = pb.u * cb.c5 + pa.u * ca.c5;
  double t7 = pb.v * cb.c5 + pa.v * ca.c5;
  double t8 = cb.c4 + ca.c4;
  double du = pb.u - pa.u, dv = pb.v - pa.v, dei = pb.e - pa.e;
  Tri f;
  f.f2 = b1 * du + b5 * dv;
  f.f3 = b5 * du + b2 * dv;
  f.f4 = (t4 + t7) * du + (t5 + t6) * dv + t8 * dei;
  return f;
}

// velocities and internal energy by division (q2/q1 ...), as the cross
// derivative terms use them
struct DivPrim { double u, v, e; };
__device__ __forceinline__ DivPrim div_prim_of(double q1, double q2, double q3, double q4) {
  DivPrim d;
  d.u = q2 / q1;
  d.v = q3 / q1;
  d.e = q4 / q1 - .5 * (sqd(d.u) + sqd(d.v));
  return d;
}
__device__ __forceinline__ DivPrim div_prim(const DevMesh& M, long long i) {
  return div_prim_of(M.q[0][i], M.q[1][i], M.q[2][i], M.q[3][i]);
}

// cross-derivative term of a line at a cell from its neighbours across the
// line: the eta line's from its j neighbours (src/visrhs.f:106-146), the xi
// line's from its k neighbours (src/visrhs.f:227-268).  The coefficients of
// the two velocity gradients change places between them.
__device__ __forceinline__ Tri vis_cross(const VisCoef& c, const DivPrim& p, const DivPrim& m, bool eta) {
  const double du = 0.5 * (p.u - m.u), dv = 0.5 * (p.v - m.v), de = 0.5 * (p.e - m.e);
  const double d5 = eta ? c.d5 : c.d7, d7 = eta ? c.d7 : c.d5;
  Tri f;
  f.f2 = c.d1 * du + d5 * dv;
  f.f3 = d7 * du + c.d2 * dv;
  double t = 0.5 * c.d1 * 0.5 * (sqd(p.u) - sqd(m.u));
  t = t + 0.5 * c.d2 * 0.5 * (sqd(p.v) - sqd(m.v));
  const double su = p.u + m.u, sv = p.v + m.v;
  t = t + c.d5 * 0.5 * (eta ? su : sv) * (eta ? dv : du);
  t = t + c.d7 * 0.5 * (eta ? sv : su) * (eta ? du : dv);
  f.f4 = t + c.d4 * de;
  return f;
}

// A workgroup owns VIS_TJ x VIS_TK interior cells.  Every per-cell quantity
// of the reference's line loops -- primitives, quotient primitives, metrics,
// the coefficients and cross terms of both directions -- is formed once for
// the cells of the tile and of its one-cell ring and kept in LDS; each cell
// then assembles its two face fluxes per direction from there.  The
// arithmetic of every quantity is the reference's, so the result does not
// depend on the tiling.
constexpr int VIS_TJ = 32, VIS_TK = 8, VIS_THREADS = VIS_TJ * VIS_TK;
constexpr int VIS_RJ = VIS_TJ + 2, VIS_RK = VIS_TK + 2;
constexpr int VIS_NR = VIS_RJ * VIS_RK;   // tile and ring, ring row 0 = k0-1, column 0 = j0-1
constexpr int VIS_NE = VIS_TJ * VIS_RK;   // eta cells: tile columns, rows k0-1 .. k0+TK
constexpr int VIS_NX = VIS_RJ * VIS_TK;   // xi cells: columns j0-1 .. j0+TJ, tile rows

// The first phase's per-cell quantities that only the coefficients read and
// the coefficients themselves share their memory: each thread holds its (at
// most VIS_PER) coefficient cells in registers across a barrier.
constexpr int VIS_PER = (VIS_NE + VIS_NX + VIS_THREADS - 1) / VIS_THREADS;
struct VisLds {
  double u[VIS_NR], v[VIS_NR], e[VIS_NR];
  union {
    struct {
      double vnu[VIS_NR], gkap[VIS_NR], du[VIS_NR], dv[VIS_NR], de[VIS_NR];
      double xx[VIS_NR], xy[VIS_NR], yx[VIS_NR], yy[VIS_NR], r[VIS_NR];
    };
    struct {
      double ec[4][VIS_NE], eg[3][VIS_NE];     // eta: c1 c2 c5 c4 and the cross term
      double xc[4][VIS_NX], xg[3][VIS_NX];     // xi
    };
    double red[4][RES_THREADS];
  };
};
constexpr size_t VIS_LDS = sizeof(VisLds);

__device__ __forceinline__ VisPrim lds_prim(const VisLds& L, int c) {
  VisPrim p;
  p.u = L.u[c]; p.v = L.v[c]; p.e = L.e[c]; p.vnu = L.vnu[c]; p.gkap = L.gkap[c];
  return p;
}
// the face fluxes read u, v and e only
__device__ __forceinline__ VisPrim lds_uve(const VisLds& L, int c) {
  VisPrim p;
  p.u = L.u[c]; p.v = L.v[c]; p.e = L.e[c]; p.vnu = 0.; p.gkap = 0.;
  return p;
}
__device__ __forceinline__ DivPrim lds_div(const VisLds& L, int c) {
  DivPrim d;
  d.u = L.du[c]; d.v = L.dv[c]; d.e = L.de[c];
  return d;
}
__device__ __forceinline__ VisMet lds_met(const VisLds& L, int c) {
  VisMet m;
  m.xx = L.xx[c]; m.xy = L.xy[c]; m.yx = L.yx[c]; m.yy = L.yy[c]; m.r = L.r[c];
  return m;
}
template <int N>
__device__ __forceinline__ VisCoef lds_coef(const double (&cf)[4][N], int c) {
  VisCoef o{};
  o.c1 = cf[0][c]; o.c2 = cf[1][c]; o.c5 = cf[2][c]; o.c4 = cf[3][c];
  return o;
}
template <int N>
__device__ __forceinline__ Tri lds_tri(const double (&g)[3][N], int c) {
  Tri f;
  f.f2 = g[0][c]; f.f3 = g[1][c]; f.f4 = g[2][c];
  return f;
}

// Bound by latency at the 12 waves a CU its LDS (41 KB) and registers (168)
// allow; FP64 issue alone is 97 us of the 60-case batch's 218 us (286 us with
// each array in memory of its own, 77 KB and 8 waves a CU); 513x129: 9.4 us
// (9.7 both ways when that was changed).
// With norms set, the residual is complete once this kernel has added the
// viscous terms, so each tile also takes its residual-norm partials here
// (the tiles and thread-to-cell map are the residual's: 32x8 tiles, k-tile
// major), instead of a separate pass over s.
__global__ __launch_bounds__(VIS_THREADS, 3) void k_visrhs(const DevMesh* __restrict__ Ms, int norms) {
  static_assert(VIS_TJ == RES_TJ && VIS_TK == RES_TK, "visrhs tiles are the residual's");
  const DevMesh& M = Ms[blockIdx.y];
  const int nj = M.je - M.js + 1, nk = M.ke - M.ks + 1;
  const int tiles_j = (nj + VIS_TJ - 1) / VIS_TJ;
  const int tile = xcd_tile(tiles_j * ((nk + VIS_TK - 1) / VIS_TK));
  if (tile < 0 || *M.status) return;
  extern __shared__ __attribute__((aligned(16))) double vis_raw[];
  VisLds& L = *reinterpret_cast<VisLds*>(vis_raw);
  const DevConst& C = M.c;
  const double gkpr = C.gamma / C.pr, prtr = C.pr / 0.9, dre = .5 / C.rey;
  const double c2b = 198.6 / C.tinf, c2bp = c2b + 1.;
  const int j0 = M.js + (tile % tiles_j) * VIS_TJ, k0 = M.ks + (tile / tiles_j) * VIS_TK;
  const int t = threadIdx.x;
  const gd_t qj = M.q[M.nq - 1];

  // tile and ring: primitives (src/visrhs.f:47-57), quotient primitives
  // (src/visrhs.f:108-119), metrics and 1/q(nq)
  for (int n = t; n < VIS_NR; n += VIS_THREADS) {
    const int j = j0 - 1 + n % VIS_RJ, k = k0 - 1 + n / VIS_RJ;
    if (j > M.je + 1 || k > M.ke + 1) continue;
    const long long i = cell(M, j, k);
    const double q1 = M.q[0][i], q2 = M.q[1][i], q3 = M.q[2][i], q4 = M.q[3][i], turm = M.turmu[i];
    const double xx = M.xx[i], xy = M.xy[i], yx = M.yx[i], yy = M.yy[i], qn = qj[i];
    const VisPrim p = vis_prim_of(q1, q2, q3, q4, turm, C.ggm1, c2b, c2bp, prtr);
    const DivPrim d = div_prim_of(q1, q2, q3, q4);
    L.u[n] = p.u; L.v[n] = p.v; L.e[n] = p.e; L.vnu[n] = p.vnu; L.gkap[n] = p.gkap;
    L.du[n] = d.u; L.dv[n] = d.v; L.de[n] = d.e;
    L.xx[n] = xx; L.xy[n] = xy; L.yx[n] = yx; L.yy[n] = yy; L.r[n] = 1. / qn;
  }
  __syncthreads();

  // coefficients and cross terms: eta along the tile columns for rows
  // k0-1 .. k0+TK, xi along the tile rows for columns j0-1 .. j0+TJ
  double oc[VIS_PER][7];
#pragma unroll
  for (int u = 0; u < VIS_PER; ++u) {
    const int n = t + VIS_THREADS * u;
    if (n >= VIS_NE + VIS_NX) break;
    const bool eta = n < VIS_NE;
    const int m = n - VIS_NE;
    const int a = eta ? n % VIS_TJ : m % VIS_RJ, b = eta ? n / VIS_TJ : m / VIS_RJ;
    if (eta ? (j0 + a > M.je || k0 - 1 + b > M.ke + 1) : (j0 - 1 + a > M.je + 1 || k0 + b > M.ke)) continue;
    // the cell, and the step to its neighbours across the line
    const int c = eta ? b * VIS_RJ + a + 1 : (b + 1) * VIS_RJ + a, d = eta ? 1 : VIS_RJ;
    const VisCoef o = vis_coef(eta ? L.yx[c] : L.xx[c], eta ? L.yy[c] : L.xy[c], L.r[c], lds_met(L, c - d),
                               lds_met(L, c + d), lds_prim(L, c), dre, gkpr);
    const Tri g = vis_cross(o, lds_div(L, c + d), lds_div(L, c - d), eta);
    oc[u][0] = o.c1; oc[u][1] = o.c2; oc[u][2] = o.c5; oc[u][3] = o.c4;
    oc[u][4] = g.f2; oc[u][5] = g.f3; oc[u][6] = g.f4;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < VIS_PER; ++u) {
    const int n = t + VIS_THREADS * u;
    if (n >= VIS_NE + VIS_NX) break;
    const int m = n - VIS_NE;
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      if (n < VIS_NE) (q < 4 ? L.ec[q & 3] : L.eg[q - 4])[n] = oc[u][q];
      else (q < 4 ? L.xc[q & 3] : L.xg[q - 4])[m] = oc[u][q];
    }
  }
  __syncthreads();

  const int a = t % VIS_TJ, b = t / VIS_TJ;
  const int j = j0 + a, k = k0 + b;
  const bool valid = j <= M.je && k <= M.ke;
  // every thread reaches the one norm_tile call below (its barriers), so
  // cells outside the grid skip the work instead of returning
  double sv[4] = {0.0, 0.0, 0.0, 0.0};
  if (valid) {
    const long long i = cell(M, j, k);
    double s2 = M.s[1][i], s3 = M.s[2][i], s4 = M.s[3][i];
    const int c = (b + 1) * VIS_RJ + a + 1;
    const VisPrim p1 = lds_uve(L, c);
    // ---- eta part (j = const line): faces k-1|k, k|k+1, cross terms
    {
      const int e = (b + 1) * VIS_TJ + a;
      const VisCoef c0 = lds_coef(L.ec, e - VIS_TJ), c1 = lds_coef(L.ec, e), c2 = lds_coef(L.ec, e + VIS_TJ);
      const Tri fm = vis_face(lds_uve(L, c - VIS_RJ), c0, p1, c1);   // face k-1
      const Tri fp = vis_face(p1, c1, lds_uve(L, c + VIS_RJ), c2);   // face k
      const Tri gm = lds_tri(L.eg, e - VIS_TJ), gc = lds_tri(L.eg, e);
      if (k < M.ke) {
        const Tri gp = lds_tri(L.eg, e + VIS_TJ);
        s2 = s2 + (fp.f2 - fm.f2) + 0.5 * (gp.f2 - gm.f2);
        s3 = s3 + (fp.f3 - fm.f3) + 0.5 * (gp.f3 - gm.f3);
        s4 = s4 + (fp.f4 - fm.f4) + 0.5 * (gp.f4 - gm.f4);
      } else {  // one-sided closure at kend (src/visrhs.f:141-150)
        Tri gq;
        if (b >= 1) {
          gq = lds_tri(L.eg, e - 2 * VIS_TJ);
        } else {  // row k-2 lies below the tile's ring
          const VisPrim pq = vis_prim(M, cell(M, j, k - 2), c2b, c2bp, prtr);
          const VisCoef cq = eta_coef(M, j, k - 2, pq, dre, gkpr);
          gq = vis_cross(cq, div_prim(M, cell(M, j + 1, k - 2)), div_prim(M, cell(M, j - 1, k - 2)), true);
        }
        s2 = s2 + (fp.f2 - fm.f2) + 0.5 * (gq.f2 - 4. * gm.f2 + 3 * gc.f2);
        s3 = s3 + (fp.f3 - fm.f3) + 0.5 * (gq.f3 - 4. * gm.f3 + 3 * gc.f3);
        s4 = s4 + (fp.f4 - fm.f4) + 0.5 * (gq.f4 - 4. * gm.f4 + 3. * gc.f4);
      }
    }
    // ---- xi part (k = const line)
    {
      const int x = b * VIS_RJ + a + 1;
      const VisCoef c0 = lds_coef(L.xc, x - 1), c1 = lds_coef(L.xc, x), c2 = lds_coef(L.xc, x + 1);
      const Tri fm = vis_face(lds_uve(L, c - 1), c0, p1, c1);
      const Tri fp = vis_face(p1, c1, lds_uve(L, c + 1), c2);
      const Tri gm = lds_tri(L.xg, x - 1), gc = lds_tri(L.xg, x);
      if (j < M.je) {
        const Tri gp = lds_tri(L.xg, x + 1);
        s2 = s2 + (fp.f2 - fm.f2) + 0.5 * (gp.f2 - gm.f2);
        s3 = s3 + (fp.f3 - fm.f3) + 0.5 * (gp.f3 - gm.f3);
        s4 = s4 + (fp.f4 - fm.f4) + 0.5 * (gp.f4 - gm.f4);
      } else {  // one-sided closure at jend (src/visrhs.f:262-271)
        Tri gq;
        if (a >= 1) {
          gq = lds_tri(L.xg, x - 2);
        } else {  // column j-2 lies left of the tile's ring
          const VisPrim pq = vis_prim(M, cell(M, j - 2, k), c2b, c2bp, prtr);
          const VisCoef cq = xi_coef(M, j - 2, k, pq, dre, gkpr);
          gq = vis_cross(cq, div_prim(M, cell(M, j - 2, k + 1)), div_prim(M, cell(M, j - 2, k - 1)), false);
        }
        s2 = s2 + (fp.f2 - fm.f2) + 0.5 * (gq.f2 - 4. * gm.f2 + 3 * gc.f2);
        s3 = s3 + (fp.f3 - fm.f3) + 0.5 * (gq.f3 - 4. * gm.f3 + 3 * gc.f3);
        s4 = s4 + (fp.f4 - fm.f4) + 0.5 * (gq.f4 - 4. * gm.f4 + 3 * gc.f4);
      }
    }
    M.s[1][i] = s2;
    M.s[2][i] = s3;
    M.s[3][i] = s4;
    sv[0] = M.s[0][i]; sv[1] = s2; sv[2] = s3; sv[3] = s4;
  }
  if (norms) {
    const ResTile T{(int)blockIdx.y, j0, k0, tile};
    __syncthreads();   // the reduction takes the coefficients' memory
    norm_tile(M, T, j, k, valid, sv, &L.red[0][0]);
  }
}

// ========================================================================= SA
// constants of src/sadata.h:2-4
constexpr double SA_cb1 = 0.1355, SA_sigma = 0.6666667, SA_cb2 = 0.622, SA_akt = 0.41,
                 SA_cw1 = 3.2390678, SA_cw2 = 0.3, SA_cw3 = 2., SA_cv1 = 7.1, SA_ct3 = 1.2, SA_ct4 = 0.5;

// integer powers as the reference build evaluates them (left to right)
__device__ __forceinline__ double ip3(double x) { return (x * x) * x; }
__device__ __forceinline__ double ip6(double x) { return ((((x * x) * x) * x) * x) * x; }

// laminar viscosity (lamvis, src/samodel2d.f:200-238) and the velocities
// vmu_sa keeps (src/samodel2d.f:61-72), all cells
// ovl: the state as ilu2d's primitive round trip leaves it
__global__ __launch_bounds__(256) void k_sa_prim(const DevMesh* __restrict__ Ms, int ovl) {
  const DevMesh& M = Ms[blockIdx.y];
  if (*M.status) return;
  long long n2 = (long long)M.jd * M.kd;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n2; i += 256ll * gridDim.x) {
    double q1 = M.q[0][i], q2 = M.q[1][i], q3 = M.q[2][i], q4 = M.q[3][i];
    if (ovl) q_roundtrip(q1, q2, q3, q4, M.q[M.nq - 1][i]);
    sa_prim_cell(M, i, q1, q2, q3, q4);
  }
}

__device__ __forceinline__ int sa_periodic_src(int idir, int js, int je, int ks, int ke, int jd, int kd, int jk) {
  if (idir == 1) { int jj = je - js + 1; return jd - 2 * jj + (jk - js + 1); }
  if (idir == -1) { int jj = je - js + 1; return 1 + 2 * jj - (je - jk + 1); }
  if (idir == 2) { int kk = ke - ks + 1; return kd - 2 * kk + (jk - ks + 1); }
  int kk = ke - ks + 1;
  return 1 + 2 * kk - (ke - jk + 1);
}

// c_turm (src/samodel2d.f:372-399) for one cell, from its q(1), q(nq),
// laminar viscosity and q(5)
__device__ __forceinline__ double c_turm_val(double q1, double qn, double vmul, double q5) {
  double rj = q1 * qn;
  double vnul = vmul / rj;
  double chi = q5 / vnul;
  double fv1 = ip3(chi) / (ip3(chi) + ip3(SA_cv1));
  return q1 * qn * q5 * fv1;
}
// the eddy viscosity of cell i; with ovl the SA model runs beside ilu2d, so
// q1 is taken through ilu2d's round trip, (q1 qj) / qj, and the value goes
// to turmu_n
__device__ __forceinline__ void put_turm(const DevMesh& M, long long i, double q1, double qj, double vmul, double q5,
                                         int ovl) {
  if (ovl) M.turmu_n[i] = c_turm_val((q1 * qj) / qj, qj, vmul, q5);
  else M.turmu[i] = c_turm_val(q1, qj, vmul, q5);
}

__device__ __forceinline__ void c_turm_cell(const DevMesh& M, long long i, int ovl) {
  put_turm(M, i, M.q[0][i], M.q[M.nq - 1][i], M.sa_vmul[i], M.q[4][i], ovl);
}

// turbc (src/samodel2d.f:827-1303) for one boundary segment
__device__ void turbc_segment(const DevMesh& M, const DevBC& b, int t, int nt) {
  const gd_t q5 = M.q[4];
  const gd_t u = M.sa_u;
  const gd_t v = M.sa_v;
  {
    int js = b.js, je = b.je, ks = b.ks, ke = b.ke, idir = b.idir;
    int iadd = idir >= 0 ? 1 : -1, iadir = idir >= 0 ? idir : -idir;
    int ty = b.type;
    double foso = 1.0;
    if (ty == 3 || ty == 4) {  // turbc_extpt, one halo layer
      if (iadir == 1) {
        int j = (idir == 1) ? je : js, j1 = j + iadd, j2 = j1 + iadd;
        for (int k = ks + t; k <= ke; k += nt)
          q5[cell(M, j, k)] = (1. + foso) * q5[cell(M, j1, k)] - foso * q5[cell(M, j2, k)];
      } else if (iadir == 2) {
        int k = (idir == 2) ? ke : ks, k1 = k + iadd, k2 = k1 + iadd;
        for (int j = js + t; j <= je; j += nt)
          q5[cell(M, j, k)] = (1. + foso) * q5[cell(M, j, k1)] - foso * q5[cell(M, j, k2)];
      }
    } else if (ty == 5) {  // turbc_wall
      if (iadir == 1) {
        int j = (idir == 1) ? je : js, j1 = j + iadd;
        for (int k = ks + t; k <= ke; k += nt) q5[cell(M, j, k)] = -q5[cell(M, j1, k)];
      } else if (iadir == 2) {
        int k = (idir == 2) ? ke : ks, k1 = k + iadd;
        for (int j = js + t; j <= je; j += nt) q5[cell(M, j, k)] = -q5[cell(M, j, k1)];
      }
    } else if (ty == 10 || ty == 11) {  // turbc_sym
      if (iadir == 1) {
        int j = (idir == 1) ? je : js, j1 = (idir == 1) ? je + 1 : js - 1;
        for (int k = ks + t; k <= ke; k += nt) q5[cell(M, j, k)] = q5[cell(M, j1, k)];
      } else if (iadir == 2) {
        int k = (idir == 2) ? ke : ks, k1 = (idir == 2) ? ke + 1 : ks - 1;
        for (int j = js + t; j <= je; j += nt) q5[cell(M, j, k)] = q5[cell(M, j, k1)];
      }
    } else if (ty == 22) {  // turbc_periodic
      int nj = je - js + 1, nk = ke - ks + 1;
      for (int w = t; w < nj * nk; w += nt) {
        int j = js + w % nj, k = ks + w / nj;
        long long src = (iadir == 1) ? cell(M, sa_periodic_src(idir, js, je, ks, ke, M.jd, M.kd, j), k)
                                     : cell(M, j, sa_periodic_src(idir, js, je, ks, ke, M.jd, M.kd, k));
        q5[cell(M, j, k)] = q5[src];
      }
    } else if (ty == 51 && iadir == 2) {  // turbc_wake
      int k = (idir == 2) ? ke : ks, k1 = (idir == 2) ? ke + 1 : ks - 1;
      for (int j = js + t; j <= je; j += nt) {
        int jj = M.jd - j + 1;
        double a = q5[cell(M, jj, k1)], c = q5[cell(M, j, k1)];
        q5[cell(M, j, k)] = a;
        q5[cell(M, jj, k)] = c;
      }
    } else if (ty == 46) {  // turbc_inf
      int nj = je - js + 1, nk = ke - ks + 1;
      for (int w = t; w < nj * nk; w += nt) q5[cell(M, js + w % nj, ks + w / nj)] = M.c.vnuinf;
    } else if (ty == 47) {  // turbc_out
      if (iadir == 1) {
        int j = (idir == 1) ? je : js, j1 = j + iadd;
        for (int k = ks + t; k <= ke; k += nt) {
          long long i = cell(M, j, k), i1 = cell(M, j1, k);
          double ug = M.has_gv ? M.ug[i] : 0.0, vg = M.has_gv ? M.vg[i] : 0.0;
          double ug1 = M.has_gv ? M.ug[i1] : 0.0, vg1 = M.has_gv ? M.vg[i1] : 0.0;
          double val = M.c.vnuinf;
          double uu = (u[i] - ug + u[i1] - ug1) * M.xx[i];
          uu = uu + (v[i] - vg + v[i1] - vg1) * M.xy[i];
          uu = uu * iadd;
          if (uu < 0.) val = q5[i1];
          q5[i] = val;
        }
      } else if (iadir == 2) {
        int k = (idir == 2) ? ke : ks, k1 = k + iadd;
        for (int j = js + t; j <= je; j += nt) {
          long long i = cell(M, j, k), i1 = cell(M, j, k1);
          double ug = M.has_gv ? M.ug[i] : 0.0, vg = M.has_gv ? M.vg[i] : 0.0;
          double ug1 = M.has_gv ? M.ug[i1] : 0.0, vg1 = M.has_gv ? M.vg[i1] : 0.0;
          double val = M.c.vnuinf;
          double uu = (u[i] - ug + u[i1] - ug1) * M.yx[i];
          uu = uu + (v[i] - vg + v[i1] - vg1) * M.yy[i];
          uu = uu * iadd;
          if (uu < 0.) val = q5[i1];
          q5[i] = val;
        }
      }
    }
  }
}

// turbc of an instance by one workgroup (the segments of a phase side by
// side).  With eddy set (the final turbc) the eddy viscosity of the halo ring
// follows (c_turm)
__global__ __launch_bounds__(BC_MAX_THREADS) void k_turbc(const DevMesh* __restrict__ Ms, int eddy, int ovl) {
  const DevMesh& M = Ms[blockIdx.x];
  if (*M.status) return;
  for_phases(M, [&](const DevBC& b, int t, int nt) { turbc_segment(M, b, t, nt); });
  if (!eddy) return;
  const int jd = M.jd, kd = M.kd;
  const int nring = 2 * jd + 2 * (kd - 2);
  for (int w = threadIdx.x; w < nring; w += (int)blockDim.x) {
    int j, k;
    if (w < jd) { j = w + 1; k = 1; }
    else if (w < 2 * jd) { j = w - jd + 1; k = kd; }
    else if (w < 2 * jd + kd - 2) { j = 1; k = w - 2 * jd + 2; }
    else { j = jd; k = w - 2 * jd - (kd - 2) + 2; }
    c_turm_cell(M, cell(M, j, k), ovl);
  }
}

// convective upwind speeds of a contravariant velocity (src/samodel2d.f:483-491)
struct UpDown { double p, m; };
__device__ __forceinline__ UpDown sa_updown(double uu) { return {0.5 * (uu + fabs(uu)), 0.5 * (uu - fabs(uu))}; }

// diffusion half-point coefficient chp and difference dnuhp of the face
// between cells with (vnul, nu-tilde) a and b (src/samodel2d.f:575-584, 622-631)
__device__ __forceinline__ void sa_half(double va, double na, double vb, double nb, double rey, double& chp,
                                        double& dn) {
  double vnulh = 0.5 * (va + vb);
  double vnuh = 0.5 * (na + nb);
  chp = (1. + SA_cb2) / SA_sigma / rey * (vnulh + vnuh);
  dn = nb - na;
}

// rhslhs (convec + diffus + source) and the pseudo-time scaling of vmu_sa
// (src/samodel2d.f:101-131, 402-824), in gather form: each cell assembles its
// own row of the two tridiagonal systems.  A workgroup takes a 32x8 tile:
// what the stencil reads of a cell (nu-tilde, vnul, contravariant velocities,
// velocities, metrics) is formed once for the tile and its one-cell ring in
// LDS.  Bound by FP64 issue (about 1100 operations a cell, 40 divisions among
// them).  60 cases (3.9 M cells): 176 us; with every thread gathering its
// neighbours' planes and forming their quantities again 256 us (two
// divisions a neighbour, 160-220 registers).  513x129: 8.3 us (9).
constexpr int SAR_N = VIS_NR;
struct SaLds {
  double nt[SAR_N], vn[SAR_N], U[SAR_N], V[SAR_N], u[SAR_N], v[SAR_N], xx[SAR_N], xy[SAR_N], yx[SAR_N], yy[SAR_N];
};

__global__ __launch_bounds__(VIS_THREADS, 4) void k_sa_rhs(const DevMesh* __restrict__ Ms) {
  __shared__ SaLds L;
  const DevMesh& M = Ms[blockIdx.y];
  const int js = M.js, je = M.je, ks = M.ks, ke = M.ke;
  const int nj = je - js + 1, nk = ke - ks + 1;
  const int tiles_j = (nj + VIS_TJ - 1) / VIS_TJ;
  const int tile = xcd_tile(tiles_j * ((nk + VIS_TK - 1) / VIS_TK));
  if (tile < 0 || *M.status) return;
  const DevConst& C = M.c;
  const double rey = C.rey;
  const int j0 = js + (tile % tiles_j) * VIS_TJ, k0 = ks + (tile / tiles_j) * VIS_TK;
  const int t = threadIdx.x;
  for (int n = t; n < SAR_N; n += VIS_THREADS) {
    const int j = j0 - 1 + n % VIS_RJ, k = k0 - 1 + n / VIS_RJ;
    if (j > je + 1 || k > ke + 1) continue;
    const long long i = cell(M, j, k);
    const double u = M.sa_u[i], v = M.sa_v[i], xx = M.xx[i], xy = M.xy[i], yx = M.yx[i], yy = M.yy[i];
    const double vmul = M.sa_vmul[i], q1 = M.q[0][i], qn = M.q[M.nq - 1][i], nt = M.q[4][i];
    const double ug = M.has_gv ? M.ug[i] : 0.0, vg = M.has_gv ? M.vg[i] : 0.0;
    L.nt[n] = nt;
    L.vn[n] = vmul / q1 / qn;
    L.U[n] = xx * (u - ug) + xy * (v - vg);
    L.V[n] = yx * (u - ug) + yy * (v - vg);
    L.u[n] = u; L.v[n] = v; L.xx[n] = xx; L.xy[n] = xy; L.yx[n] = yx; L.yy[n] = yy;
  }
  __syncthreads();
  const int j = j0 + t % VIS_TJ, k = k0 + t / VIS_TJ;
  if (j <= je && k <= ke) {
    const long long i = cell(M, j, k);
    const int c = (t / VIS_TJ + 1) * VIS_RJ + t % VIS_TJ + 1, w = c - 1, e = c + 1, s = c - VIS_RJ, n = c + VIS_RJ;
    const double nt = L.nt[c], vnul = L.vn[c];
    const double xx = L.xx[c], xy = L.xy[c], yx = L.yx[c], yy = L.yy[c];
    // ---- convec (src/samodel2d.f:493-538)
    double sj = M.s[4][i];
    double aj = 0.0, bj = 0.0, cj = 0.0, ak = 0.0, bk = 0.0, ck = 0.0;
    const UpDown cu = sa_updown(L.U[c]), cv = sa_updown(L.V[c]);
    sj = sj - cu.p * (nt - L.nt[w]) - cu.m * (L.nt[e] - nt);
    sj = sj - cv.p * (nt - L.nt[s]) - cv.m * (L.nt[n] - nt);
    if (j > js) {
      const UpDown x = sa_updown(L.U[w]);
      aj = aj - (cu.p > 1.0e-12 ? 1.0 : 0.0) * (x.p + x.m);
    }
    bj = bj + cu.p - cu.m;
    if (j < je) {
      const UpDown x = sa_updown(L.U[e]);
      cj = cj + (cu.m < -1.0e-12 ? 1.0 : 0.0) * (x.p + x.m);
    }
    if (k > ks) {
      const UpDown x = sa_updown(L.V[s]);
      ak = ak - (cv.p > 1.0e-12 ? 1.0 : 0.0) * (x.p + x.m);
    }
    bk = bk + cv.p - cv.m;
    if (k < ke) {
      const UpDown x = sa_updown(L.V[n]);
      ck = ck + (cv.m < -1.0e-12 ? 1.0 : 0.0) * (x.p + x.m);
    }
    // ---- diffus, j direction (src/samodel2d.f:570-607)
    {
      double chpm, dnm, chpp, dnp;
      sa_half(L.vn[w], L.nt[w], vnul, nt, rey, chpm, dnm);
      sa_half(vnul, nt, L.vn[e], L.nt[e], rey, chpp, dnp);
      double dmxhm = 0.5 * (L.xx[w] + xx), dmyhm = 0.5 * (L.xy[w] + xy);
      double dmxhp = 0.5 * (xx + L.xx[e]), dmyhp = 0.5 * (xy + L.xy[e]);
      double dxp = dmxhp * xx + dmyhp * xy;
      double dxm = dmxhm * xx + dmyhm * xy;
      double c2 = SA_cb2 / SA_sigma / rey;
      c2 = c2 * (vnul + nt);
      double dcp = dxp * (chpp - c2);
      double dcm = dxm * (chpm - c2);
      double ax = fmax(dcm, 0.0), cx = fmax(dcp, 0.0);
      sj = sj - ax * dnm + cx * dnp;
      aj = aj - ax;
      cj = cj - cx;
      bj = bj + ax + cx;
    }
    // ---- diffus, k direction (src/samodel2d.f:617-654)
    {
      double chpm, dnm, chpp, dnp;
      sa_half(L.vn[s], L.nt[s], vnul, nt, rey, chpm, dnm);
      sa_half(vnul, nt, L.vn[n], L.nt[n], rey, chpp, dnp);
      double dmxhm = 0.5 * (L.yx[s] + yx), dmyhm = 0.5 * (L.yy[s] + yy);
      double dmxhp = 0.5 * (yx + L.yx[n]), dmyhp = 0.5 * (yy + L.yy[n]);
      double dyp = dmxhp * yx + dmyhp * yy;
      double dym = dmxhm * yx + dmyhm * yy;
      double c2 = SA_cb2 / SA_sigma / rey;
      c2 = c2 * (vnul + nt);
      double dcp = dyp * (chpp - c2);
      double dcm = dym * (chpm - c2);
      double ay = fmax(dcm, 0.0), cy = fmax(dcp, 0.0);
      sj = sj - ay * dnm + cy * dnp;
      ak = ak - ay;
      ck = ck - cy;
      bk = bk + ay + cy;
    }
    // ---- source (src/samodel2d.f:729-811), isour = 0, fturf = 0
    {
      double vort = 0.0;
      if (M.bodyflag) {
        double ux = (L.u[e] - L.u[w]) * 0.5;
        double vx = (L.v[e] - L.v[w]) * 0.5;
        double uy = (L.u[n] - L.u[s]) * 0.5;
        double vy = (L.v[n] - L.v[s]) * 0.5;
        vort = fabs(xy * ux - xx * vx + yy * uy - yx * vy);
      }
      const double d2min = 1.e-12, rmax = 10.0, stilim = 1.e-12, fturf = 0.0;
      const double cv1_3 = ip3(SA_cv1), cw3_6 = ip6(SA_cw3);
      double chi = nt / vnul;
      double d = M.sa_sn[i];
      chi = fmax(chi, 1.e-12);
      double chi3 = ip3(chi);
      double fv1 = chi3 / (chi3 + cv1_3);
      double fv2 = 1. - chi / (1. + chi * fv1);
      double fv3 = 1.0;
      double ft2 = fturf * SA_ct3 * exp(-1. * SA_ct4 * chi * chi);
      double dchi = 1. / vnul;
      double dfv1 = (3. * cv1_3) * (chi * chi) * dchi * sqd(1. / (chi3 + cv1_3));
      double dfv2 = (fv2 - 1.) / chi / vnul + (1. - fv2) * (1 - fv2) * (dfv1 + fv1 / chi / vnul);
      double dfv3 = 0.0;
      double dft2 = (-2. * SA_ct4) * chi * dchi * ft2;
      double d2 = fmax(d * d, d2min);
      double stilda = vort * fv3 + vnul / (d2 * SA_akt * SA_akt * rey) * chi * fv2;
      stilda = fmax(stilda, stilim);
      double r = nt / (d2 * SA_akt * SA_akt * rey) / stilda;
      r = fmin(r, rmax);
      double g = r + SA_cw2 * (ip6(r) - r);
      double g6 = ip6(g);
      double fw = (1. + cw3_6) / (g6 + cw3_6);
      fw = g * pow(fw, 1. / 6.);
      double dstild = vort * dfv3 + vnul * (dchi * fv2 + chi * dfv2) / (d2 * SA_akt * SA_akt * rey);
      double dr = vnul * (dchi - chi * dstild / stilda) / stilda / (d2 * SA_akt * SA_akt * rey);
      double dg = dr * (1. + SA_cw2 * (6. * pow(r, 5.) - 1.));
      double dfw = pow((1. + cw3_6) / (g6 + cw3_6), 1. / 6.);
      dfw = dfw * dg * (1. - g6 / (g6 + cw3_6));
      double pro = SA_cb1 * stilda * (1. - ft2);
      double des = (SA_cw1 * fw - SA_cb1 / (SA_akt * SA_akt) * ft2) / d2 / rey;
      double prod = SA_cb1 * stilda * (1. - ft2) * nt;
      double dest = (SA_cw1 * fw - SA_cb1 / (SA_akt * SA_akt) * ft2) * nt * nt / d2 / rey;
      double dpro = pro * dstild / stilda - SA_cb1 * stilda * dft2;
      double ddes = (SA_cw1 * dfw - SA_cb1 / (SA_akt * SA_akt) * dft2) / d2 / rey * vnul * chi;
      ddes = ddes + des;
      ddes = ddes * nt;
      dpro = dpro * nt;
      sj = sj + prod - dest;
      double tk1 = fmax(des * nt - pro, 0.0);
      double tk2 = fmax(ddes - dpro, 0.0);
      bk = bk + tk1 + tk2;
    }
    // ---- scale by the turbulence pseudo time step
    double tscal = M.tscale[i];
    if (C.timeac == 1.) {
      double qj = M.q[M.nq - 1][i];
      tscal = (double)imx(M.iblank[i], 0) * (1.0 + 0.002 * sqrt(qj)) / (1. + sqrt(qj));
      tscal = tscal * 1.0;
      tscal = tscal / (1. + tscal / C.h);
    }
    M.sa_sj[i] = sj * tscal;
    M.sa_aj[i] = aj * tscal;
    M.sa_cj[i] = cj * tscal;
    M.sa_ak[i] = ak * tscal;
    M.sa_ck[i] = ck * tscal;
    M.sa_bb[i] = 1. + (bj + bk) * tscal;
  }
}

// The two scalar tridiagonal solves of vmu_sa (lsolvej, lsolvek), each line
// solved in parts (part_line, part_columns).
// lsolvej (src/samodel2d.f:1306-1344) and s1, sjmat*bjmat of vmu_sa
// (src/samodel2d.f:148-152) for the k row blockIdx.x, one wave.
// Bound by one memory round trip and the parts' chain at one case (513x129:
// 5.3 us; by two lanes from both ends out of LDS 37 us), by HBM in a batch
// (60 cases, 3.9 M cells, 40 bytes a cell: 38 us; one lane per line side, 99 us).
__global__ __launch_bounds__(64) void k_sa_solve_j(const DevMesh* __restrict__ Ms) {
  __shared__ __attribute__((aligned(16))) double buf[PART_BUF];
  const DevMesh& M = Ms[blockIdx.y];
  if (*M.status) return;
  const int k = M.ks + blockIdx.x;
  if (k > M.ke) return;
  const long long i0 = cell(M, M.js, k);
  part_line(gptr(M.sa_aj) + i0, gptr(M.sa_bb) + i0, gptr(M.sa_cj) + i0, gptr(M.sa_sj) + i0, M.je - M.js + 1, buf);
}

// lsolvek (src/samodel2d.f:1347-1385), s2 and the nu-tilde update with its
// clip (src/samodel2d.f:157-188), then the interior eddy viscosity (c_turm)
// for TC adjacent j columns.  8 columns are half a 128-byte line; with the
// neighbouring workgroup on the same XCD the other half comes out of its L2,
// and twice the workgroups of 16 columns hide more latency: 60 cases 94 us;
// with empty workgroups among them 102 (16 columns 111, 4 columns 126; 8 without
// the runs per XCD 137; lane per line and an update pass of its own 125), 20
// cases 35 (16: 37).  513x129 7.7 (16: 8.8, 4: 7.6; two lanes per column from
// both ends 17.4).
constexpr int SAK_NT = 512;
template <int TC>
__global__ __launch_bounds__(SAK_NT) void k_sa_solve_k(const DevMesh* __restrict__ Ms, int ovl) {
  extern __shared__ __attribute__((aligned(16))) double sak_ex[];
  constexpr int PM = PCOL_M;
  const DevMesh& M = Ms[blockIdx.y];
  if (*M.status) return;
  const int group = xcd_tile((M.je - M.js + TC) / TC);
  if (group < 0) return;
  const int j0 = M.js + group * TC;
  const int n = M.ke - M.ks + 1, P = (n + PM - 1) / PM;
  const int j = j0 + (int)threadIdx.x % TC, k0 = ((int)threadIdx.x / TC) * PM;
  const bool col = j <= M.je;
  const long long st = M.jd, i0 = cell(M, col ? j : M.je, M.ks);
  const gdouble *ga = gptr(M.sa_ak), *gb = gptr(M.sa_bb), *gc = gptr(M.sa_ck), *gs = gptr(M.sa_sj);
  double a[PM], b[PM], c[PM], s[PM];
#pragma unroll
  for (int u = 0; u < PM; ++u) {
    const long long i = i0 + (long long)(k0 + u < n ? k0 + u : n - 1) * st;
    a[u] = ga[i]; b[u] = gb[i]; c[u] = gc[i]; s[u] = gs[i];
  }
#pragma unroll
  for (int u = 0; u < PM; ++u) {
    const int k = k0 + u;
    if (k >= n) { a[u] = 0.; b[u] = 1.; s[u] = 0.; }
    if (k == 0) a[u] = 0.;
    if (k >= n - 1) c[u] = 0.;
  }
  // the update's operands, ahead of the solve
  const double vnulim = 1.0e-20, relfac = 1.0;
  const gdouble *g5 = gptr(M.q[4]), *g1 = gptr(M.q[0]), *gj = gptr(M.q[M.nq - 1]), *gv = gptr(M.sa_vmul);
  double q5[PM], q1[PM], qj[PM], vm[PM];
  int ib[PM];
#pragma unroll
  for (int u = 0; u < PM; ++u) {
    const long long i = i0 + (long long)(k0 + u < n ? k0 + u : n - 1) * st;
    q5[u] = g5[i]; q1[u] = g1[i]; qj[u] = gj[i]; vm[u] = gv[i]; ib[u] = M.iblank[i];
  }
  part_columns<TC>(a, b, c, s, P, sak_ex);
#pragma unroll
  for (int u = 0; u < PM; ++u) {
    if (!col || k0 + u >= n) continue;
    const long long i = i0 + (long long)(k0 + u) * st;
    const double dq = relfac * (0. + s[u]);
    const double v = fmax((q5[u] + dq * (double)imx(ib[u], 0)), vnulim);
    M.q[4][i] = v;
    put_turm(M, i, q1[u], qj[u], vm[u], v, ovl);
  }
}

// distance to the wall (dist, src/samodel2d.f:243-293); static grids: once
__global__ __launch_bounds__(256) void k_sa_dist(const DevMesh* __restrict__ Ms) {
  const DevMesh& M = Ms[blockIdx.y];
  const int jd = M.jd, kd = M.kd;
  long long n2 = (long long)jd * kd;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n2; i += 256ll * gridDim.x) {
    int j = 1 + (int)(i % jd), k = 1 + (int)(i / jd);
    double sn = 1.e10;
    if (M.bodyflag) {
      if (j >= M.jtail1 && j <= M.jtail2) {
        if (k == 1) sn = 0.0;
        else {
          int jv = j - 1;
          sn = sqrt(sqd(M.x[i] - 0.5 * (M.xv[vert(M, jv, 1)] + M.xv[vert(M, jv + 1, 1)])) +
                    sqd(M.y[i] - 0.5 * (M.yv[vert(M, jv, 1)] + M.yv[vert(M, jv + 1, 1)])));
        }
      } else {
        int jv = M.jtail1 - 1;
        sn = sqrt(sqd(M.x[i] - M.xv[vert(M, jv, 1)]) + sqd(M.y[i] - M.yv[vert(M, jv, 1)]));
      }
    }
    M.sa_sn[i] = sn;
  }
}

static inline int nblk2(long long n, int per) {
  long long b = (n + per - 1) / per;
  return (int)(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

static long long max_cells(const DevMesh* hM, int nmi) {
  long long mx = 0;
  for (int i = 0; i < nmi; ++i) mx = hM[i].jd * (long long)hM[i].kd > mx ? hM[i].jd * (long long)hM[i].kd : mx;
  return mx;
}

// As many waves for each segment of an instance's largest phase as its longest
// segment fills, 256 to 1024 threads in all.  Waves beyond that hold a CU
// without work while other instances of the batch wait for one: the two calls
// of a step, 1000 cases of 33x17, SA 11.5 and 12.3 us (1024 threads: 19.6 and
// 19.8), SST 14.1 and 15.0 (34.5 and 31.9); 1000 cases of 65x33, SA 14.9 and
// 17.2 (21.4 and 23.9).  From about 129 columns on it is 1024 as before.
int bc_threads(const DevMesh* hM, int nmi) {
  int waves = BC_THREADS / 64;
  for (int i = 0; i < nmi; ++i)
    for (int ph = 0; ph < hM[i].nbc_phase; ++ph) {
      int m = 0, longest = 0;
      for (int ib = 0; ib < hM[i].nbc; ++ib) {
        const DevBC& b = hM[i].bc[ib];
        if (b.phase != ph) continue;
        const int cells = (b.je - b.js + 1) * (b.ke - b.ks + 1);
        longest = cells > longest ? cells : longest;
        ++m;
      }
      const int w = m * ((longest + 63) / 64);
      waves = w > waves ? w : waves;
    }
  return 64 * waves < BC_MAX_THREADS ? 64 * waves : BC_MAX_THREADS;
}

// 32x8 tiles of the largest instance
static int vis_tiles(const DevMesh* hM, int nmi) {
  int tiles = 1;
  for (int i = 0; i < nmi; ++i) {
    const int nj = hM[i].je - hM[i].js + 1, nk = hM[i].ke - hM[i].ks + 1;
    const int n = ((nj + VIS_TJ - 1) / VIS_TJ) * ((nk + VIS_TK - 1) / VIS_TK);
    tiles = n > tiles ? n : tiles;
  }
  return tiles;
}

hipError_t launch_visrhs(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st, int norms) {
  const int tiles = vis_tiles(hM, nmi);
  static bool lds_set = false;
  if (!lds_set) {
    hipError_t e = hipFuncSetAttribute((const void*)k_visrhs, hipFuncAttributeMaxDynamicSharedMemorySize, (int)VIS_LDS);
    if (e != hipSuccess) return e;
    lds_set = true;
  }
  hipLaunchKernelGGL(k_visrhs, dim3(tiles, nmi), dim3(VIS_THREADS), VIS_LDS, st, dM, norms);
  return hipGetLastError();
}

hipError_t launch_sa_dist(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st) {
  hipLaunchKernelGGL(k_sa_dist, dim3(nblk2(max_cells(hM, nmi), 256), nmi), dim3(256), 0, st, dM);
  return hipGetLastError();
}

hipError_t launch_sa_prim(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st) {
  hipLaunchKernelGGL(k_sa_prim, dim3(nblk2(max_cells(hM, nmi), 256), nmi), dim3(256), 0, st, dM, 0);
  return hipGetLastError();
}

// vmu_sa for every instance (src/samodel2d.f:2-197, itrans = 0)
hipError_t launch_sa(const DevMesh* dM, const DevMesh* hM, int nmi, Marks* mk, hipStream_t st, int sa_lane,
                     int prim_done, int ovl) {
  long long mx = max_cells(hM, nmi);
  int mj = 1, mk_ = 1;
  for (int i = 0; i < nmi; ++i) {
    mj = hM[i].je - hM[i].js + 1 > mj ? hM[i].je - hM[i].js + 1 : mj;
    mk_ = hM[i].ke - hM[i].ks + 1 > mk_ ? hM[i].ke - hM[i].ks + 1 : mk_;
  }
  hipError_t e = hipSuccess;
  if (!prim_done) {
    hipLaunchKernelGGL(k_sa_prim, dim3(nblk2(mx, 256), nmi), dim3(256), 0, st, dM, ovl);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  mark(mk, OT2D_ST_SA_PRIM, st);
  const int nbc = bc_threads(hM, nmi);
  hipLaunchKernelGGL(k_turbc, dim3(nmi), dim3(nbc), 0, st, dM, 0, ovl);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  mark(mk, OT2D_ST_SA_BC, st);
  hipLaunchKernelGGL(k_sa_rhs, dim3(vis_tiles(hM, nmi), nmi), dim3(VIS_THREADS), 0, st, dM);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  mark(mk, OT2D_ST_SA_RHS, st);
  hipLaunchKernelGGL(k_sa_solve_j, dim3(mk_, nmi), dim3(64), 0, st, dM);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  mark(mk, OT2D_ST_SA_SOLVE_J, st);
  const int np = (mk_ + PCOL_M - 1) / PCOL_M;   // parts of the longest column
  // 8 columns a workgroup; 16 where the launch choice asks for them and they
  // fit 512 threads (columns of up to 256 cells).  Figures at k_sa_solve_k.
  const bool wide = np * 16 <= SAK_NT && sa_lane == 0;
  auto solve_k = [&](auto kern, int tc) {
    const int nt = (np * tc + 63) / 64 * 64;
    hipLaunchKernelGGL(kern, dim3((mj + tc - 1) / tc, nmi), dim3(nt), sizeof(double) * 6 * nt, st, dM, ovl);
  };
  if (wide) solve_k(k_sa_solve_k<16>, 16);
  else solve_k(k_sa_solve_k<8>, 8);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  mark(mk, OT2D_ST_SA_SOLVE_K, st);
  hipLaunchKernelGGL(k_turbc, dim3(nmi), dim3(nbc), 0, st, dM, 1, ovl);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  mark(mk, OT2D_ST_SA_EDDY, st);
  return hipSuccess;
}

}  // namespace ot2d
