// Device-side data structures shared by the gfx950 kernels and the C-ABI
// host code of libot2d.
//
// State layout in HBM is the reference's own (src/step.f:17-29): per mesh,
// Fortran column-major cell arrays (jd,kd) with j fastest, one halo ring,
// variables of q and s as separate planes q(jd,kd,nspec,nq).  A DevMesh
// record describes one (mesh, time instance) pair: base pointers already
// offset to the instance, so every kernel works on flat j-fastest planes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ot2d.h"
#include "ot2d_plain.h"

#define OT2D_MAXQ 8
// longest grid line (interior cells) of the turbulence-model line solves
#define SA_LINE_MAX 1024
#define OT2D_MAXBC_DEV 25

namespace ot2d {

// One boundary segment with the reference's index fix-ups already applied
// (src/bc.f:21-35): js..je, ks..ke are 1-based cell indices incl. halo.
struct DevBC {
  int type, idir, js, je, ks, ke;
  // segments of one phase touch disjoint cells and run side by side; the
  // phases run in order, so segments that share cells keep the reference's
  // segment order
  int phase;
};

// Case constants derived as read_inputs does (src/setup.f:1162-1248) plus
// the scheme switches the kernels branch on.
constexpr int OT2D_MAX_ITN = 16;   // Newton sub-iterations per time step, at most

struct DevConst {
  double gamma, gm1, ggm1, einf, pinf, rinf, uinf, vinf, rey, rmue, h;
  double th, qt, epse, Mp, dualtime, timeac, jac_factor, pr, tinf;
  double vnuinf, rotf;
  double tkeinf, tomegainf;  // SST free stream (src/setup.f:1232-1234)
  double angmax, xac, yac;   // time-spectral pitching (src/setup.f:348-393)
  double fmm, half, ca, sa;  // force normalisation (src/forces.f:27-31, 166-172)
  int invisc, iread, ilim, iconstant_cfl, idual, iprecon, timespectral, ntac;
  int iturb, nmv, motiontype;
  int itnmax;                // Newton sub-iterations per time step
  int iunst;                 // 1: the grid pitches every time step (motiontype 1)
  double dtps[OT2D_MAX_ITN]; // dtpseudo(itn), the dual time of sub-iteration itn
};

// A pointer into device memory held in a record: subscripts go through the
// global address space.  A plain pointer loaded from a record is generic to
// the compiler: its accesses become flat instructions, which count against
// the LDS counter as well and whose completions are only known together, so
// loads issued ahead do not stay in flight.
template <typename T>
struct GPtr {
  typedef __attribute__((address_space(1))) T G;
  T* p;
  __host__ __device__ GPtr& operator=(T* q) { p = q; return *this; }
  __host__ __device__ operator T*() const { return p; }
  template <typename I>
  __device__ __forceinline__ G& operator[](I i) const { return ((G*)p)[i]; }
  __device__ __forceinline__ G& operator*() const { return *(G*)p; }
  template <typename I>
  __device__ __forceinline__ GPtr operator+(I i) const { GPtr r; r.p = p + i; return r; }
};
typedef GPtr<double> gd_t;

struct DevMesh {
  int jd, kd, jmax, kmax;
  int js, je, ks, ke;        // jbeg, jend, kbeg, kend (1-based)
  int nq, nv, nbc, nspec, nsp;
  int nbc_phase;             // phases of the boundary segments
  int jtail1, jtail2;
  int has_gv;                // grid velocities present (time-spectral)
  int res_block0, res_nblocks;  // this instance's slice of the norm partials
  double epsj, epsk;         // Koren limiter epsilons (src/eulerrhs.f:51-52)
  DevBC bc[OT2D_MAXBC_DEV];
  GPtr<double> q[OT2D_MAXQ];  // q(:,:,nsp,n) planes, n = 1..nq  (index n-1)
  GPtr<double> s[OT2D_MAXQ];  // s(:,:,nsp,n) planes
  GPtr<double> x, y, xx, xy, yx, yy, ug, vg, turmu, tscale, bt;
  GPtr<double> turmu_n;  // SA beside ilu2d: the new eddy viscosity until the update takes it
  GPtr<double> xv, yv, ugv, vgv;  // vertex arrays (jmax,kmax) of this instance
  GPtr<const double> xv0, yv0;  // instance-1 vertices (time-spectral rotation)
  GPtr<double> xold, yold, xole, yole;  // vertices one and two time steps back (moving grids), or null
  GPtr<int> iblank;
  int bodyflag;              // mesh has a wall segment (type 5)
  // SA workspace (jd,kd) planes: laminar viscosity, u, v, wall distance and
  // the rows of the two tridiagonal systems (src/samodel2d.f:22-30)
  GPtr<double> sa_vmul, sa_u, sa_v, sa_sn, sa_sj, sa_aj, sa_cj, sa_ak, sa_ck, sa_bb;
  // SST workspace (src/komegasst.f:20-41): F1, F2*rho*strain/Re, production,
  // cross diffusion, and per equation (k, omega) the rows of the j and k
  // tridiagonal systems sharing one diagonal
  GPtr<double> kw_f1, kw_x, kw_prod, kw_cd;
  GPtr<double> kw_s[2], kw_a[2], kw_b[2], kw_c[2], kw_ak[2], kw_ck[2];
  GPtr<double> lu;  // LU-SGS sweep records (workspace)
  int lu_fp32;               // sweep arithmetic: 1 FP32, 0 FP64
  // per-case bookkeeping (shared by all instances of a case)
  GPtr<int> status;  // 0 ok, 1 mstop, 2 norm
  GPtr<int> istep0;  // device copy of istep0
  GPtr<int> istep;  // time steps of this run (the driver's istep; time-accurate steps)
  GPtr<double> ta;  // time-accurate levels: qtn, qtnm1, qnewt (nv planes each), or null
  GPtr<double> partials;  // norm partials of this instance's tiles (res_nblocks * 4 doubles)
  GPtr<double> norms;  // rsum, resrho, resmax, jmax, kmax, nmax
  GPtr<int> stepc;  // steps started in the current ot2d_iterate call
  GPtr<double> hist;  // residual history rsum[step][slot] (may be null)
  int hist_cap, hist_stride, hist_slot;
  GPtr<double> tspec;  // time instant of this instance
  GPtr<const double> Ds;  // spectral derivative matrix (nspec x nspec)
  GPtr<double> qall[OT2D_MAXQ];  // q planes of instance 0 (TS coupling base)
  long long inst_stride;     // elements between instances within a plane set
  DevConst c;
};

// Residual work item: one TJ x TK tile of interior cells of one instance.
struct ResTile {
  int mesh;   // index into the DevMesh array
  int j0, k0; // first interior cell (1-based)
  int blk;    // tile index within the instance (norm partial slot)
};

// plain global-address-space pointers, for the arguments of line solves
typedef __attribute__((address_space(1))) double gdouble;
__device__ __forceinline__ gdouble* gptr(const gd_t& p) { return (gdouble*)p.p; }

// ------------------------------------------------- turbulence line solves
// One line of contiguous cells by one wave (lane = part): the four arrays
// come in coalesced and pass through LDS (`buf`, PART_BUF doubles) to the
// lanes' parts, then y = x * b goes back the same way into s.
constexpr int PART_BUF = 64 * 18;
template <int M>
__device__ __forceinline__ void part_line_wave(const gdouble* ga, const gdouble* gb, const gdouble* gc, gdouble* gs,
                                               int n, double* buf) {
  constexpr int LD = M + 2;   // a lane's cells in LDS: 16-byte reads, no bank conflicts
  typedef double d2_t __attribute__((ext_vector_type(2)));
  const int l = threadIdx.x & 63;
  const int P = (n + M - 1) / M;
  double v[4][M];
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int e = l + 64 * u, ec = e < n ? e : n - 1;
    v[0][u] = ga[ec]; v[1][u] = gb[ec]; v[2][u] = gc[ec]; v[3][u] = gs[ec];
  }
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int e = l + 64 * u;
    if (e >= n) { v[0][u] = 0.; v[1][u] = 1.; v[3][u] = 0.; }
    if (e == 0) v[0][u] = 0.;
    if (e >= n - 1) v[2][u] = 0.;
  }
  // one wave's LDS operations run in order: no barrier
  auto transpose = [&](double (&x)[M]) {
#pragma unroll
    for (int u = 0; u < M; ++u) {
      const int e = l + 64 * u;
      buf[e / M * LD + e % M] = x[u];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int u = 0; u < M; u += 2) {
      const d2_t t = *reinterpret_cast<const d2_t*>(buf + l * LD + u);
      x[u] = t.x; x[u + 1] = t.y;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
#pragma unroll
  for (int q = 0; q < 4; ++q) transpose(v[q]);
  double (&a)[M] = v[0], (&b)[M] = v[1], (&c)[M] = v[2], (&s)[M] = v[3];
  part_eliminate<M>(a, b, c, s);
  auto down = [&](double x, int d) { const double y = __shfl_down(x, d); return l + d < 64 ? y : 0.; };
  auto up = [&](double x, int d) { const double y = __shfl_up(x, d); return l >= d ? y : 0.; };
  SepRow w = part_separator<M>(a, b, c, s, down(s[0], 1), down(a[0], 1), down(c[0], 1));
  for (int d = 1; d < P; d <<= 1) {
    const SepRow m = {up(w.A, d), up(w.C, d), up(w.D, d)}, p = {down(w.A, d), down(w.C, d), down(w.D, d)};
    w = sep_reduce(w, m, p);
  }
  part_expand<M>(a, c, s, up(w.D, 1), w.D);
#pragma unroll
  for (int u = 0; u < M; ++u) s[u] = (0. + s[u] - 0.) * b[u];
#pragma unroll
  for (int u = 0; u < M; u += 2) *reinterpret_cast<d2_t*>(buf + l * LD + u) = d2_t{s[u], s[u + 1]};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int e = l + 64 * u;
    if (e < n) gs[e] = buf[e / M * LD + e % M];
  }
}
__device__ __forceinline__ void part_line(const gdouble* a, const gdouble* b, const gdouble* c, gdouble* s, int n,
                                          double* buf) {
  switch (part_cells(n)) {
    case 8: part_line_wave<8>(a, b, c, s, n, buf); break;
    case 12: part_line_wave<12>(a, b, c, s, n, buf); break;
    default: part_line_wave<16>(a, b, c, s, n, buf); break;
  }
}

// TC adjacent columns of n <= 512 rows by one workgroup: thread (column c =
// tid % TC, part p = tid / TC) holds rows 8p .. 8p+7 of its column, so every
// load of a wave is whole row segments of TC cells.  The separators' rows
// pass between the parts through LDS (`ex`, two buffers of 3 x threads).
// On return s holds x.  Every thread of the workgroup calls it.
constexpr int PCOL_M = 8;
template <int TC>
__device__ __forceinline__ void part_columns(double (&a)[PCOL_M], const double (&b)[PCOL_M], double (&c)[PCOL_M],
                                             double (&s)[PCOL_M], int P, double* ex) {
  constexpr int M = PCOL_M;
  const int nt = blockDim.x, tid = threadIdx.x, p = tid / TC;
  part_eliminate<M>(a, b, c, s);
  double* e0 = ex;
  double* e1 = ex + 3 * nt;
  auto post = [&](double x, double y, double z) { e0[tid] = x; e0[nt + tid] = y; e0[2 * nt + tid] = z; };
  auto at = [&](int q) -> SepRow {   // the row of part q of this column
    const int o = tid + (q - p) * TC;
    const bool in = q >= 0 && q < P;
    const int oc = in ? o : tid;
    const double x = e0[oc], y = e0[nt + oc], z = e0[2 * nt + oc];
    return {in ? x : 0., in ? y : 0., in ? z : 0.};
  };
  auto swap = [&]() { double* t = e0; e0 = e1; e1 = t; };
  post(s[0], a[0], c[0]);
  __syncthreads();
  const SepRow nx = at(p + 1);
  swap();
  SepRow w = part_separator<M>(a, b, c, s, nx.A, nx.C, nx.D);
  for (int d = 1; d < P; d <<= 1) {
    post(w.A, w.C, w.D);
    __syncthreads();
    const SepRow m = at(p - d), q = at(p + d);
    swap();
    w = sep_reduce(w, m, q);
  }
  e0[tid] = w.D;
  __syncthreads();
  const double XL = p > 0 ? e0[tid - TC] : 0.;
  swap();
  part_expand<M>(a, c, s, XL, w.D);
}

// Tile of this workgroup among the n of its record, or -1: xcd_deal.  Against
// tiles in dispatch order: 385x97 with 401x401, FP32 operators 27.7 -> 23.6
// us, viscous terms 23.5 -> 21.5; 60 cases: viscous terms 231 -> 223, residual
// 260 -> 254, SA right-hand side 189 -> 182 (with launches filled up to a
// multiple of 8 a record; without, 21.9 and 18.9, 218, 254 and 176).
__device__ __forceinline__ int xcd_tile(int n) { return xcd_deal((int)blockIdx.x, n); }

constexpr int RES_TJ = 32;
constexpr int RES_TK = 8;
constexpr int RES_THREADS = RES_TJ * RES_TK;

// The turbulence models' boundary conditions and those of the residual run
// one workgroup per instance.  The segments of a phase touch disjoint cells:
// f(segment, t, nt) runs for as many of them side by side as there are waves,
// each on a group of whole waves (t, nt: the thread's number in its group and
// the group's size); the phases follow one another with a barrier between.
constexpr int BC_THREADS = 256, BC_MAX_THREADS = 1024;
template <typename F>
__device__ __forceinline__ void for_phases(const DevMesh& M, F f) {
  const int nw = (int)(blockDim.x >> 6);
  for (int ph = 0; ph < M.nbc_phase; ++ph) {
    int m = 0;   // segments of this phase
    for (int ib = 0; ib < M.nbc; ++ib) m += M.bc[ib].phase == ph;
    for (int g0 = 0; g0 < m; g0 += nw) {
      const int groups = m - g0 < nw ? m - g0 : nw, nt = 64 * (nw / groups);
      const int mine = __builtin_amdgcn_readfirstlane((int)threadIdx.x / nt);
      if (mine < groups) {
        int q = g0 + mine, ib = 0;
        for (;; ++ib)
          if (M.bc[ib].phase == ph && q-- == 0) break;
        f(M.bc[ib], (int)threadIdx.x - mine * nt, nt);
      }
    }
    __syncthreads();
  }
}

// oat of the time-accuracy order (src/time.f:22-25): the reference's istep
// counts the time steps of the run
__device__ inline double time_oat(const DevMesh& M) {
  double oat = 1.0;
  if (M.c.ntac < 2) return oat;
  const int istep = *M.istep;
  if (M.c.ntac >= 2 && istep > 1) oat = 2. / 3.;
  if (M.c.ntac == 3 && istep > 2) oat = 6. / 11.;
  return oat;
}

// round trip of ilu2d's in-place primitive conversion (src/lhs.f:524-531,
// 805-811): the reference leaves q(j,k,1:4) with these bits
__device__ __forceinline__ void q_roundtrip(double& q1, double& q2, double& q3, double& q4, double qj) {
  double dj = 1.0 / q1;
  double u = q2 * dj, v = q3 * dj, e = q4 * dj;
  double r = q1 * qj;
  q1 = r / qj;
  q2 = u * q1; q3 = v * q1; q4 = e * q1;
}

// laminar viscosity (lamvis, src/samodel2d.f:200-238) and the velocities
// vmu_sa keeps (src/samodel2d.f:61-72) of one cell from its state
__device__ inline void sa_prim_cell(const DevMesh& M, long long i, double q1, double q2, double q3, double q4) {
  const double c2b = 198.6 / M.c.tinf, c2bp = c2b + 1.;
  double ra = 1. / q1;
  double uvel = q2 * ra, vvel = q3 * ra;
  double ei = q4 * ra - 0.5 * (uvel * uvel + vvel * vvel);
  double tt = M.c.ggm1 * ei;
  M.sa_vmul[i] = c2bp * tt * sqrt(tt) / (c2b + tt);
  M.sa_u[i] = q2 / q1;
  M.sa_v[i] = q3 / q1;
}

__host__ __device__ inline long long cell(const DevMesh& M, int j, int k) {
  return (long long)(j - 1) + (long long)(k - 1) * M.jd;
}

// residual norms of step (src/step.f:53-115), first stage: the partial sums
// (sum of squares, rho part, max |s| with its first (k,n,j) position) of the
// cells of one tile, reduced in a fixed order and stored per tile
__device__ inline void norm_tile(const DevMesh& M, const ResTile& T, int j, int k, bool valid, const double* s,
                                 double* redbuf) {
  double(*red)[RES_THREADS] = reinterpret_cast<double(*)[RES_THREADS]>(redbuf);
  const int tid = threadIdx.x;
  const int jd = M.jd;
  double rs = 0.0, rr1 = 0.0, rmax = 0.0, key = 0.0;
  if (valid) {
    long long i = cell(M, j, k);
    double ibp = (double)(M.iblank[i] > 0 ? M.iblank[i] : 0);
    double m1 = s[0] * ibp, m2 = s[1] * ibp, m3 = s[2] * ibp, m4 = s[3] * ibp;
    rs = m1 * m1 + m2 * m2 + m3 * m3 + m4 * m4;
    rr1 = s[0] * s[0];
    // first maximum in (k, n, j) order (src/step.f:67-78)
    for (int n = 0; n < 4; ++n) {
      double a = fabs(s[n]) * ibp;
      if (a > rmax) { rmax = a; key = (double)(((long long)(k - 1) * 4 + n) * jd + (j - 1)); }
    }
  }
  if (tid < RES_THREADS) {   // threads past the tile's cells pass the barriers only
    red[0][tid] = rs; red[1][tid] = rr1; red[2][tid] = rmax; red[3][tid] = valid && rmax > 0.0 ? key : 1e300;
  }
  __syncthreads();
  for (int off = RES_THREADS / 2; off > 0; off >>= 1) {
    if (tid < off) {
      red[0][tid] = red[0][tid] + red[0][tid + off];
      red[1][tid] = red[1][tid] + red[1][tid + off];
      double a = red[2][tid], b = red[2][tid + off];
      double ka = red[3][tid], kb = red[3][tid + off];
      if (b > a || (b == a && kb < ka)) { red[2][tid] = b; red[3][tid] = kb; }
    }
    __syncthreads();
  }
  if (tid == 0) {
    const gd_t P = M.partials + 4ll * T.blk;
    P[0] = red[0][0]; P[1] = red[1][0]; P[2] = red[2][0]; P[3] = red[3][0];
  }
}
__host__ __device__ inline long long vert(const DevMesh& M, int j, int k) {
  return (long long)(j - 1) + (long long)(k - 1) * M.jmax;
}

}  // namespace ot2d

// launch wrappers (ot2d_kernels.hip)
namespace ot2d {
// Optional per-kernel HIP events for profiling: mark(m, s, st) is recorded on
// the launch stream right after the kernel of stage s (an OT2D_ST_* value).
struct Marks {
  static constexpr int CAP = 64;
  hipEvent_t ev[CAP];
  int stage[CAP];
  int n = 0;
};
inline void mark(Marks* m, int s, hipStream_t st) {
  if (m && m->n < Marks::CAP) {
    (void)hipEventRecord(m->ev[m->n], st);
    m->stage[m->n++] = s;
  }
}

hipError_t launch_init_geometry(const DevMesh* dM, int nmi, hipStream_t st);
// metfv alone on moved vertices (no cell centres, no free-stream state), as
// the time loop of a moving grid does
hipError_t launch_metrics(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
// pitch (src/motion.f:546-632): the grid turns by this time step's angle
hipError_t launch_pitch(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
// with ncase > 0 also opens the step of every running case (istep0 and the
// step counter)
hipError_t launch_time_step(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st, int* istep0 = nullptr,
                            const int* status = nullptr, int* stepc = nullptr, int ncase = 0, int itn = 0);
// time-accurate steps with Newton sub-iterations (src/time.f:109-209)
hipError_t launch_open_step(const int* status, int* istep0, int* stepc, int* istep, int ncase, hipStream_t st);
hipError_t launch_stqol(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
hipError_t launch_newton(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
hipError_t launch_copy_doubles(double* dst, const double* src, int n, hipStream_t st);
hipError_t launch_bc(const DevMesh* dM, const DevMesh* hM, int nmi, int zero_s, hipStream_t st);
hipError_t launch_residual(const DevMesh* dM, const ResTile* tiles, int ntiles, int do_norms, int weno,
                           hipStream_t st);
hipError_t launch_norms(const DevMesh* dM, const ResTile* tiles, int ntiles, hipStream_t st);
// rbc: the residual boundary conditions follow in the same launch
hipError_t launch_norms_final(const DevMesh* dM, int nmi, hipStream_t st, int rbc = 0);
hipError_t launch_conv_check(const DevMesh* dM, const int* inst, const double* tol, int* status, int ncase,
                             hipStream_t st);
hipError_t launch_rbc(const DevMesh* dM, int nmi, hipStream_t st);
// threads of a workgroup that runs an instance's turbulence boundary conditions
int bc_threads(const DevMesh* hM, int nmi);
// launch choices that change no result (the autotuner's knobs)
constexpr int LU_R = 32;   // rows of one LU-SGS sweep workgroup (two lanes per row)
constexpr int LU32_SWEEP_VARIANTS = 3;   // FP32 sweep instantiations (ring steps, producers, prefetch)
// Version of what the numbers of a LaunchCfg stand for, part of the key that
// choices are cached under (also in files): raised with every change of an
// instantiation behind a number.
constexpr int LAUNCH_SET = 2;
struct LaunchCfg {
  int sweep = 0;     // 0: 15 ring steps, 3 producers; 1: 18, 3; 2: 12, 4 (with deeper prefetch)
  int sa_lane = -1;  // SA k solves: columns per workgroup, 0: 16, 1 and -1: 8
};
// fuse_update: 1 the q update and monitor in k_lu_finish (Euler), | 2
// k_lu_finish also leaves the turbulence models' laminar viscosity and
// velocities (what k_sa_prim computes) from the state it writes
hipError_t launch_lu(const DevMesh* dM, const DevMesh* hM, int nmi, int fuse_update, int fp32, Marks* mk,
                     hipStream_t st, int sweep = 0);
hipError_t launch_monitor(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
hipError_t launch_update_monitor(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st, int take_turmu = 0);
// k_lu_finish alone (launch_lu with fuse_update | 4 leaves it out)
hipError_t launch_lu_finish(const DevMesh* dM, const DevMesh* hM, int nmi, int flags, int fp32, hipStream_t st);
hipError_t launch_forces(const DevMesh* dM, int mi, double* out, hipStream_t st);
hipError_t launch_tsrhs(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
// bytes of one instance's LU-SGS workspace (rl: ceil(rows / 64) of the case's
// tallest mesh, part of the size rule of batch slots)
size_t lu_workspace_bytes(int jd, int kd, int rl);
hipError_t launch_visrhs(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st, int norms = 0);
// prim_done: the laminar viscosity and velocities are already in place
// (k_lu_finish with flag 2)
// ovl: the SA model runs beside ilu2d (another stream, before k_lu_finish):
// it takes q1-q4 through ilu2d's primitive round trip itself and leaves the
// eddy viscosity in turmu_n, which k_update_monitor copies
hipError_t launch_sa(const DevMesh* dM, const DevMesh* hM, int nmi, Marks* mk, hipStream_t st, int sa_lane = -1,
                     int prim_done = 0, int ovl = 0);
hipError_t launch_sa_dist(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
hipError_t launch_sa_prim(const DevMesh* dM, const DevMesh* hM, int nmi, hipStream_t st);
hipError_t launch_sst(const DevMesh* dM, const DevMesh* hM, int nmi, Marks* mk, hipStream_t st, int prim_done = 0);
// overset interpolation (ot2d_overset.hip): don/fr are device arrays of
// {int mi, jj, kk, pad; double f1, f2} and {int mi, jj, kk, src}
hipError_t launch_interp(const DevMesh* dM, const void* don, int ndon, const void* fr, int nfr, double* qbc, int nv,
                         hipStream_t st);
size_t interp_donor_bytes();
size_t interp_fringe_bytes();
// longest j line (interior cells) a case may have: what the sweeps' staging
// in LDS once allowed, kept as the library's limit (the sweeps stage nothing
// by line length; at 512 rows their records end well inside 32-bit offsets)
int lu_max_ni(int fp32);
}  // namespace ot2d
