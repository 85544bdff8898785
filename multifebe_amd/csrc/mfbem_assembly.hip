// BEM influence-matrix assembly on MI355X (gfx950), FP64.
//
// Pipeline of one mesh (all kernels on one stream):
//   mesh creation (geometry only, once):
//     k_elem_setup     per element: characteristic length, gln_far, bounding ball
//     k_precalc        per element x precalculated point: x, n, phi*J*w for Gauss-Legendre 2..9
//     k_node_normals   per node: normalised sum of element normals (ctype 10 loads)
//     k_classify       per element block x collocation nodes: integration class of every pair
//     k_fill_lists     pair ids grouped by class (precalculated rule r, adaptive, singular),
//                      each class list ordered by element so that batches share element data
//     k_sing_geom, k_adapt_geom  what the singular and the adaptive pairs take from the geometry
//   every assembly (material / frequency dependent):
//     k_begin<T>       b := 0 and the few entries of A that no tile stores
//     k_regular_tile<H> one wave per tile of up to 16 pairs of one element and one precalculated
//                      rule, one launch per element colour: kernel values straight into the FP64
//                      matrix cores, the first colour of a node stores, the others add
//     k_fold_extra<T>  rows of the second points of edge nodes added to their nodes' rows
//     k_near<H>        adaptive pairs (a wave each), singular pairs (a workgroup each) and free
//                      terms (a thread each) in one launch, added atomically
//   k_regular<H>       per-rule variant writing per-pair blocks
//   k_field, k_points  interior displacements of the precalculated pairs
// Scatter follows the BE-ordinary rule of src/assemble_bem_{staela,harela}_equation.f90: the
// unknown of node j, direction k is column 3j+k; u-known directions move h to b and put -g in A.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <complex>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "mfbem.h"
#include "mfbem_device.h"
#include "mfbem_internal.h"

namespace mfb {

__constant__ GLTables c_gl;
__device__ inline const GLTables& gl() { return c_gl; }

// Polar sub-triangles of a collocation point on one of the 9 nodes of a quad9 (nodal collocation:
// every singular pair has its point there).  Computed once on the host, whose libm is the one the
// reference calls: the number of angular points, 5 + nint(25 dtheta / (pi/2)), sits exactly on a
// half-integer at corner nodes (dtheta = pi/4) and a 1-ulp difference in asin flips it.
struct PolarSet {
  int n;
  int st[8];
  int ngt[8];
  double th[16];
  double thp[16];
};
__constant__ PolarSet c_polar[9];
// Their quadrature points, (xi1, xi2, rho x weights) each: they depend on the node alone, so a
// singular pair reads them instead of taking tan, atan, sine and cosine per point.
constexpr int kPolarMax = 2400;  // 8 sub-triangles of at most 20 x 15 points
__device__ double g_polar_pts[9][kPolarMax][3];
__constant__ int c_polar_np[9];

constexpr int kWave = 64;
// deepest adaptive subdivision
constexpr int kMaxNs = 20;
// largest precalculated rule: g^2 points x 360 B of kernel values and weights (harmonic) within
// the 160 KB of LDS a gfx950 workgroup may hold
constexpr int kMaxPrecalGln = 21;
constexpr size_t kMaxLds = 160 * 1024;
constexpr int kMaxIncid = 24;

// Collocation points: the reference's nodal SBIE puts one point on every node; a node on the open
// edge of a boundary (an element edge with no neighbour) is collocated by SBIE-MCA instead, with
// one point inside every element that holds the node, all adding to the node's equations
// (src/assign_default_bem_formulation.f90:74-93, src/build_lse_mechanics_bem_staela.f90:890-925).
// Pairs are (collocation point cp, element e), pair id e * ncp + cp.
struct DevMesh {
  int nn, ne, n_ps, npts;  // npts: precalculated points per element (sum of gln^2)
  int ncp;                 // collocation points
  int ps_gln[kMaxPrecalsets], ps_off[kMaxPrecalsets + 1];
  int ns_max;
  double qsi_re, tol;
  const double* x;
  const int* conn;
  const int* ctype;
  const double* cval;
  const double* elem;  // 8 per element: cl, radius, centre(3), gln_far, 0, 0
  const double* ps;    // (ne, npts, kPsStride)
  const double* nfn;   // (nn, 3)
  const int* inc_ptr;  // node -> (element, local node) incidences, ordered by element
  const int* inc_e;
  const int* inc_k;
  const double* xc;             // (ncp, 3) collocation point coordinates
  const int* crow;              // (ncp) node whose equations (rows 3 crow + l) the point adds to
  // (ncp) MCA points that share their node's rows with an earlier point have rows of their own, 3 cx ..
  // 3 cx + 2 of an extra matrix of 3 nx rows (TileOut::X); -1: the rows of A
  const int* cx;
  const int* xnode;             // (nx) node of each extra point, ascending
  int nx;
  const int* cel;               // (ncp) element holding an MCA point, -1 for a nodal point
  const double* cxi;            // (ncp, 2) local coordinates of an MCA point in cel
  const unsigned char* nmca;    // (nn) 1 for a node collocated by MCA points
  const unsigned char* ekind;   // (ne) kNeedH | kNeedG: kernels that element's conditions need
  const int* enode;             // (ne, 9) node; ~node where an element of a lower colour holds it
  const int2* emask;            // (ne) bit 3 n + k of node n, direction k: u prescribed; value not zero
};

// What an element contributes: with h (t*) to columns of unknown u and, where u is prescribed and not
// zero, to b; with g (u*) to columns of unknown t and, where t is prescribed and not zero, to b.  A
// traction-free element needs h alone, one held at zero g alone.
// kTwice: the element holds a node more than once (its columns then meet in one instruction).
constexpr int kNeedH = 1, kNeedG = 2, kTwice = 4;

// ------------------------------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------------------------------
template <bool H>
struct Val;
template <>
struct Val<false> {
  typedef double T;
};
template <>
struct Val<true> {
  typedef zd T;
};

__device__ inline void atomic_add(double* a, double v) { unsafeAtomicAdd(a, v); }
__device__ inline void atomic_add(zd* a, zd v) {
  unsafeAtomicAdd(&a->re, v.re);
  unsafeAtomicAdd(&a->im, v.im);
}
__device__ inline double mag(double a) { return fabs(a); }
__device__ inline double mag(zd a) { return hypot(a.re, a.im); }
__device__ inline double zero_of(double) { return 0.0; }
__device__ inline zd zero_of(zd) { return mkz(0.0); }
template <typename T>
__device__ inline T from_real(double v);
template <>
__device__ inline double from_real<double>(double v) { return v; }
template <>
__device__ inline zd from_real<zd>(double v) { return mkz(v); }
__device__ inline double scale_h(const KernelParams& k, double v) { return v * k.ctet1; }
__device__ inline double scale_g(const KernelParams& k, double v) { return v * k.cteu1; }
__device__ inline zd scale_h(const KernelParams& k, zd v) { return mkz(k.h.cte_t[0], k.h.cte_t[1]) * v; }
__device__ inline zd scale_g(const KernelParams& k, zd v) { return mkz(k.h.cte_u[0], k.h.cte_u[1]) * v; }

// Exterior kernel values at one point before the constants (bem_staela3d.f90:636-645;
// bem_harela3d.f90:657-690), h += ft*phi*jw, g += fu*phi*jw, written component by component into an
// LDS row: row[c] = ft, row[9 + c] = fu (entries `stride` apart).
__device__ inline void ext_kernel_row(const KernelParams& k, const double* x, const double* n,
                                      const double* x_i, double* row, int stride = 1) {
  double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  double r = sqrt(dot3(rv, rv)), d1r = 1.0 / r, d1r2 = d1r * d1r;
  double dr[3] = {rv[0] * d1r, rv[1] * d1r, rv[2] * d1r};
  double drdn = dot3(dr, n);
  for (int il = 0; il < 3; il++)
    for (int ik = 0; ik < 3; ik++) {
      double dk = il == ik ? 1.0 : 0.0;
      row[stride * (9 + 3 * il + ik)] = d1r * (k.cteu2 * dk + dr[il] * dr[ik]);
      row[stride * (3 * il + ik)] = d1r2 * ((k.ctet2 * dk + 3.0 * dr[il] * dr[ik]) * drdn +
                                            k.ctet2 * (n[il] * dr[ik] - n[ik] * dr[il]));
    }
}

__device__ inline void ext_kernel_row(const KernelParams& k, const double* x, const double* n,
                                      const double* x_i, zd* row, int stride = 1) {
  double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  double r, d1r;
  dist_and_inverse(dot3(rv, rv), r, d1r);
  double dr[3] = {rv[0] * d1r, rv[1] * d1r, rv[2] * d1r};
  double drdn = dot3(dr, n);
  zd psi, chi, TT1, TT2, TT3;
  har_factors<true, true>(&k.h, r, d1r, true, psi, chi, TT1, TT2, TT3);
  for (int il = 0; il < 3; il++)
    for (int ik = 0; ik < 3; ik++) {
      double dk = il == ik ? 1.0 : 0.0;
      row[stride * (9 + 3 * il + ik)] = psi * dk - chi * dr[il] * dr[ik];
      row[stride * (3 * il + ik)] = TT1 * dr[il] * dr[ik] * drdn +
                                    TT2 * (drdn * dk + dr[ik] * n[il]) + TT3 * dr[il] * n[ik];
    }
}

// Third output of the integration kernels: the displacement at interior points,
// u_l(x) = sum over pairs (x, e) of g(n, l, k) t_k(node n) - h(n, l, k) u_k(node n)
// (src/calculate_internal_points_mechanics_static.f90:76-89, ..._bem_harela.f90:355-363): the
// pair's 9x3x3 blocks are contracted with the boundary values as they are integrated.
template <typename T>
struct VecOut {
  const T* u;  // (nn, 3) boundary displacements
  const T* t;  // (nn, 3) boundary tractions
  T* out;      // (ncp, 3) interior displacements (accumulated)
};


// mesh setup and classification decide rules: plain FP64 rounding, as in the geometry helpers
#pragma clang fp contract(off)

// ------------------------------------------------------------------------------------------------
// mesh setup kernels
// ------------------------------------------------------------------------------------------------
__device__ inline void load_X(const DevMesh& m, int e, double* X) {
  for (int k = 0; k < 9; k++) {
    int j = m.conn[9 * e + k];
    for (int c = 0; c < 3; c++) X[3 * k + c] = m.x[3 * j + c];
  }
}

// fbem_qs_phijac_ngp_2d (quasisingular_integration.f90:812-975) for quad9 geometry and functions
__device__ int phijac_ngp_q9(const double* X, double eh) {
  const GLTables& G = gl();
  double leh = eh <= 0 ? 1e-6 : (eh < 1e-12 ? 1e-12 : eh);
  double in[9] = {0}, old[9];
  int j = 1;
  bool cont = true;
  while (cont) {
    for (int l = 0; l < 9; l++) { old[l] = in[l]; in[l] = 0; }
    for (int k1 = 0; k1 < j; k1++)
      for (int k2 = 0; k2 < j; k2++) {
        double d1[9], d2[9], p[9], T1[3] = {0, 0, 0}, T2[3] = {0, 0, 0}, N[3];
        dphi_q9(G.x11[j][k1], G.x11[j][k2], d1, d2);
        for (int l = 0; l < 9; l++)
          for (int c = 0; c < 3; c++) {
            T1[c] += d1[l] * X[3 * l + c];
            T2[c] += d2[l] * X[3 * l + c];
          }
        cross3(T1, T2, N);
        double jw = sqrt(dot3(N, N)) * G.w11[j][k1] * G.w11[j][k2];
        phi_q9(G.x11[j][k1], G.x11[j][k2], p);
        for (int l = 0; l < 9; l++) in[l] += (p[l] + 1.0) * jw;
      }
    if (j == 1) {
      j++;
    } else {
      cont = false;
      for (int l = 0; l < 9; l++)
        if (fabs((old[l] - in[l]) / in[l]) > leh) { cont = true; j++; break; }
      if (j == 33) cont = false;
    }
  }
  return j - 1;
}

// fbem_geometry_element_ball (geometry.f90:3904-4235), quad branch
__device__ void ball_q9(const double* X, int glp, double* centre, double* radius) {
  const GLTables& G = gl();
  double es = 0, xm[3] = {0, 0, 0};
  for (int k1 = 0; k1 < glp; k1++)
    for (int k2 = 0; k2 < glp; k2++) {
      double x[3], T1[3], T2[3], N[3];
      q9_geom(X, G.x11[glp][k1], G.x11[glp][k2], x, T1, T2);
      cross3(T1, T2, N);
      double jw = sqrt(dot3(N, N)) * G.w11[glp][k1] * G.w11[glp][k2];
      es += jw;
      for (int c = 0; c < 3; c++) xm[c] += x[c] * jw;
    }
  for (int c = 0; c < 3; c++) centre[c] = xm[c] / es;
  double r = 0;
  for (int k = 0; k < 9; k++) {
    double v[3] = {X[3 * k] - centre[0], X[3 * k + 1] - centre[1], X[3 * k + 2] - centre[2]};
    double t = sqrt(dot3(v, v));
    if (r < t) r = t;
  }
  for (int k1 = 0; k1 < glp; k1++)
    for (int k2 = 0; k2 < glp; k2++) {
      double x[3];
      q9_x(X, G.x11[glp][k1], G.x11[glp][k2], x);
      double v[3] = {x[0] - centre[0], x[1] - centre[1], x[2] - centre[2]};
      double t = sqrt(dot3(v, v));
      if (r < t) r = t;
    }
  *radius = r;
}

__global__ void k_elem_setup(DevMesh m, double* elem) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m.ne) return;
  double X[27], c[3], r;
  load_X(m, e, X);
  double cl = clen_q9(X, 1e-9);
  int nphi = phijac_ngp_q9(X, m.qsi_re);
  ball_q9(X, nphi, c, &r);
  // shape descriptors for the learned rule choice: aspect = longest / shortest edge (arc length);
  // curvature = largest |d2x/dxi2| at the centre (x7 - 2 x8 + x5, x4 - 2 x8 + x6) over cl
  double lmin = 1e300, lmax = 0;
  for (int k = 0; k < 4; k++) {
    double ye[9];
    for (int j = 0; j < 3; j++)
      for (int q = 0; q < 3; q++) ye[3 * j + q] = X[3 * kEdgeQ9[k][j] + q];
    const double le = length_l3(ye, 1e-9);
    lmin = fmin(lmin, le);
    lmax = fmax(lmax, le);
  }
  double c1 = 0, c2 = 0;
  for (int q = 0; q < 3; q++) {
    const double a = X[21 + q] - 2.0 * X[24 + q] + X[15 + q];
    const double b = X[12 + q] - 2.0 * X[24 + q] + X[18 + q];
    c1 += a * a;
    c2 += b * b;
  }
  double* o = elem + 8 * (long long)e;
  o[0] = cl; o[1] = r; o[2] = c[0]; o[3] = c[1]; o[4] = c[2]; o[5] = (double)nphi;
  o[6] = lmax / fmax(lmin, 1e-300);
  o[7] = sqrt(fmax(c1, c2)) / cl;
}

// precalculated datasets, quad branch of init_precalculated_datasets (bem_general.f90:462-530)
__global__ void k_precalc(DevMesh m, double* ps) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)m.ne * m.npts) return;
  int e = (int)(t / m.npts), q = (int)(t % m.npts);
  int r = 0;
  while (q >= m.ps_off[r + 1]) r++;
  int g = m.ps_gln[r], kt = q - m.ps_off[r], k1 = kt / g, k2 = kt % g;
  const GLTables& G = gl();
  double X[27], x[3], T1[3], T2[3], N[3], p[9];
  load_X(m, e, X);
  double x1 = G.x11[g][k1], x2 = G.x11[g][k2], w1 = G.w11[g][k1], w2 = G.w11[g][k2];
  q9_geom(X, x1, x2, x, T1, T2);
  cross3(T1, T2, N);
  double j = sqrt(dot3(N, N));
  phi_q9(x1, x2, p);
  double* o = ps + t * kPsStride;
  for (int c = 0; c < 3; c++) { o[c] = x[c]; o[3 + c] = N[c] / j; }
  for (int n = 0; n < 9; n++) o[6 + n] = p[n] * j * w1 * w2;
  o[15] = 0;
}

__global__ void k_node_normals(DevMesh m, double* nfn) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.nn) return;
  double s[3] = {0, 0, 0};
  for (int q = m.inc_ptr[i]; q < m.inc_ptr[i + 1]; q++) {
    double X[27], x[3], T1[3], T2[3], N[3];
    load_X(m, m.inc_e[q], X);
    int k = m.inc_k[q];
    q9_geom(X, kXiQ9[k][0], kXiQ9[k][1], x, T1, T2);
    cross3(T1, T2, N);
    double j = sqrt(dot3(N, N));
    for (int c = 0; c < 3; c++) s[c] += N[c] / j;
  }
  double j = sqrt(dot3(s, s));
  for (int c = 0; c < 3; c++) nfn[3 * i + c] = s[c] / j;
}

// Integration class of pair (i, e): the decision sequence of fbem_bem_staela3d_sbie_auto
// (bem_staela3d.f90:549-587), which the harmonic version repeats (bem_harela3d.f90:1498-1536).
// (all lanes of the wave call; the result of an inactive one is not used)
__device__ int classify_pair(const DevMesh& m, const QsiParams& qsp, const double* X,
                             const double* el, const double* x_i, bool active) {
  double rr[3] = {el[2] - x_i[0], el[3] - x_i[1], el[4] - x_i[2]};
  double rmin = sqrt(dot3(rr, rr)) - el[1], barxi[2] = {0, 0}, d = rmin / el[0];
  const bool near = !(rmin > 4.0 * el[1]);
  nearest_q9_wave<false>(active && near, X, el[0], x_i, barxi, &rmin, &d);
  if (near && d <= 1e-12) return m.n_ps + 1;
  int gln_near = qs_estimate(qsp, 0, 2, 5, d, barxi);
  int gln = max((int)el[5], gln_near);
  int gmax = m.ps_gln[m.n_ps - 1];
  if (gln <= gmax && gln_near > 0) {
    for (int r = 0; r < m.n_ps; r++)
      if (m.ps_gln[r] >= gln) return r;
  }
  return m.n_ps;
}

// Features of a pair for the learned rule choice (MFB_QNET_INPUTS floats):
//   log10(d) / 2 with d as sbie_auto defines it (ball distance over cl for far pairs, nearest
//   point distance over cl otherwise), log2(aspect), curvature, k cl / 4, max(|barxi_1|, |barxi_2|)
__device__ void pair_features(const double* X, const double* el, const double* x_i, double kw,
                              bool active, float* f) {
  double rr[3] = {el[2] - x_i[0], el[3] - x_i[1], el[4] - x_i[2]};
  double rmin = sqrt(dot3(rr, rr)) - el[1], barxi[2] = {0, 0}, d = rmin / el[0];
  nearest_q9_wave<false>(active && !(rmin > 4.0 * el[1]), X, el[0], x_i, barxi, &rmin, &d);
  if (!active) return;
  f[0] = (float)(0.5 * log10(fmax(d, 1e-12)));
  f[1] = (float)log2(el[6]);
  f[2] = (float)el[7];
  f[3] = (float)(0.25 * kw * el[0]);
  f[4] = (float)fmax(fabs(barxi[0]), fabs(barxi[1]));
}

__global__ void __launch_bounds__(256) k_pair_features(DevMesh m, const int* pairs, int np, double kw, float* feats) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int pid = pairs[min(q, np - 1)], e = pid / m.ncp, cp = pid % m.ncp;
  double X[27], el[8];
  load_X(m, e, X);
  for (int c = 0; c < 8; c++) el[c] = m.elem[8 * e + c];
  pair_features(X, el, m.xc + 3 * cp, kw, q < np, feats + (long long)q * MFB_QNET_INPUTS);
}

// features of every pair (pair id = e * ncp + cp), k h left at 0 (set per assembly by k_set_kh)
__global__ void __launch_bounds__(256) k_all_features(DevMesh m, float* feats) {
  const long long own = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long last = (long long)m.ne * m.ncp - 1, pid = own < last ? own : last;
  const int e = (int)(pid / m.ncp), cp = (int)(pid % m.ncp);
  double X[27], el[8];
  load_X(m, e, X);
  for (int c = 0; c < 8; c++) el[c] = m.elem[8 * e + c];
  pair_features(X, el, m.xc + 3 * cp, 0.0, own <= last, feats + pid * MFB_QNET_INPUTS);
}

__global__ void k_set_kh(DevMesh m, float* feats, double kw) {
  const long long pid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (pid >= (long long)m.ne * m.ncp) return;
  feats[pid * MFB_QNET_INPUTS + 3] = (float)(0.25 * kw * m.elem[8 * (pid / m.ncp)]);
}

// integration class of every pair from the network's class (singular pairs keep theirs): class c <
// MFB_QNET_CLASSES - 1 -> the smallest precalculated rule of order >= c + 2, moved on to promo[]
// of that rule (the judge's promotions; identity without); otherwise, or when no precalculated
// rule is that long, the adaptive rule.  counts: pairs per (element, class).
__global__ void __launch_bounds__(256) k_learned_map(DevMesh m, const unsigned char* cls_ref,
                                                     const int* qcls, const int* promo,
                                                     unsigned char* lcls, int* counts) {
  const int e = blockIdx.x;
  __shared__ int hist[kMaxPrecalsets + 2];
  if (threadIdx.x < kMaxPrecalsets + 2) hist[threadIdx.x] = 0;
  __syncthreads();
  for (int cp = threadIdx.x; cp < m.ncp; cp += blockDim.x) {
    const long long pid = (long long)e * m.ncp + cp;
    int c = cls_ref[pid];
    if (c != m.n_ps + 1) {
      const int q = qcls[pid];
      c = m.n_ps;
      if (q < MFB_QNET_CLASSES - 1)
        for (int r = 0; r < m.n_ps; r++)
          if (m.ps_gln[r] >= q + 2) { c = promo[r]; break; }
    }
    lcls[pid] = (unsigned char)c;
    atomicAdd(&hist[c], 1);
  }
  __syncthreads();
  if (threadIdx.x < m.n_ps + 2) counts[(long long)e * (kMaxPrecalsets + 2) + threadIdx.x] = hist[threadIdx.x];
}

// pairs at positions pos[k] of a list
__global__ void k_gather_list(const int* lists, const long long* pos, int k, int* out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < k) out[q] = lists[pos[q]];
}

__global__ void __launch_bounds__(256) k_classify(DevMesh m, const QsiParams* __restrict__ qsp_p,
                                                  unsigned char* cls, int* counts) {
  const QsiParams& qsp = *qsp_p;
  const int e = blockIdx.x;
  __shared__ int hist[kMaxPrecalsets + 2];
  if (threadIdx.x < kMaxPrecalsets + 2) hist[threadIdx.x] = 0;
  __syncthreads();
  double X[27], el[8];
  load_X(m, e, X);
  for (int c = 0; c < 8; c++) el[c] = m.elem[8 * e + c];
  for (int c0 = 0; c0 < m.ncp; c0 += blockDim.x) {
    const int cp = c0 + threadIdx.x;
    const int c = classify_pair(m, qsp, X, el, m.xc + 3 * min(cp, m.ncp - 1), cp < m.ncp);
    if (cp >= m.ncp) continue;
    cls[(long long)e * m.ncp + cp] = (unsigned char)c;
    atomicAdd(&hist[c], 1);
  }
  __syncthreads();
  if (threadIdx.x < m.n_ps + 2) counts[(long long)e * (kMaxPrecalsets + 2) + threadIdx.x] = hist[threadIdx.x];
}

// pair ids e*ncp+cp into per-class lists; offsets[e*(kMaxPrecalsets+2)+c] is where element e's
// pairs of class c start.  Inside an (element, class) run the points keep their order (wave ballots
// and per-wave prefix counts, no atomics), so a run of consecutive points has consecutive rows.
__global__ void __launch_bounds__(256) k_fill_lists(DevMesh m, const unsigned char* cls,
                                                    const long long* offsets, int* lists) {
  constexpr int S = kMaxPrecalsets + 2, W = 256 / kWave;
  const int e = blockIdx.x, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  __shared__ int cursor[S];
  __shared__ int wcnt[W][S];
  if (threadIdx.x < S) cursor[threadIdx.x] = 0;
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int c0 = 0; c0 < m.ncp; c0 += 256) {
    const int cp = c0 + threadIdx.x;
    const int c = cp < m.ncp ? cls[(long long)e * m.ncp + cp] : -1;
    int mine = 0;
    for (int q = 0; q < m.n_ps + 2; q++) {
      const unsigned long long mask = __ballot(c == q);
      if (c == q) mine = __popcll(mask & below);
      if (lane == 0) wcnt[wave][q] = __popcll(mask);
    }
    __syncthreads();
    if (c >= 0) {
      int pos = cursor[c] + mine;
      for (int w = 0; w < wave; w++) pos += wcnt[w][c];
      lists[offsets[(long long)e * S + c] + pos] = e * m.ncp + cp;
    }
    __syncthreads();
    if (threadIdx.x < m.n_ps + 2) {
      int t = 0;
      for (int w = 0; w < W; w++) t += wcnt[w][threadIdx.x];
      cursor[threadIdx.x] += t;
    }
    __syncthreads();
  }
}

// Tiles of the scatter kernel (k_regular_tile): element e's run of precalculated rule c is cut
// into tiles of at most kTileP consecutive list entries; toff[e*(kMaxPrecalsets+2)+c] is the
// run's first tile.  A tile is (first list entry, count, rule, element).
constexpr int kTileP = 16;
__global__ void k_fill_tiles(DevMesh m, const int* counts, const long long* offsets,
                             const long long* toff, int4* tiles) {
  constexpr int S = kMaxPrecalsets + 2;
  const int e = blockIdx.x;
  for (int c = 0; c < m.n_ps; c++) {
    const long long k = (long long)e * S + c;
    const int cnt = counts[k];
    const long long o = offsets[k], t0 = toff[k];
    for (int j = threadIdx.x; j * kTileP < cnt; j += blockDim.x)
      tiles[t0 + j] = make_int4((int)(o + (long long)j * kTileP), min(kTileP, cnt - j * kTileP), c, e);
  }
}

// classes of listed pairs only (a batch of independent pairs)
__global__ void __launch_bounds__(128) k_classify_listed(DevMesh m, const QsiParams* __restrict__ qsp_p, const int* pids,
                                  int np, unsigned char* cls) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int pid = pids[min(q, np - 1)], e = pid / m.ncp, cp = pid % m.ncp;
  double X[27], el[8];
  load_X(m, e, X);
  for (int c = 0; c < 8; c++) el[c] = m.elem[8 * e + c];
  const int c = classify_pair(m, *qsp_p, X, el, m.xc + 3 * cp, q < np);
  if (q < np) cls[q] = (unsigned char)c;
}

#pragma clang fp contract(fast)

// ------------------------------------------------------------------------------------------------
// assembly kernels
// ------------------------------------------------------------------------------------------------
__global__ void k_reset(long long* counters, int* err) {
  if (threadIdx.x < 2) counters[threadIdx.x] = 0;
  if (threadIdx.x == 0) *err = 0;
}

template <typename T>
__global__ void k_zero(T* A, long long lda, int n) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long total = (long long)n * n;
  if (lda == n) {   // contiguous: a flat fill, no index division
    for (; t < total; t += (long long)gridDim.x * blockDim.x) A[t] = zero_of(T());
  } else {
    for (; t < total; t += (long long)gridDim.x * blockDim.x) {
      long long col = t / n, row = t % n;
      A[row + lda * col] = zero_of(T());
    }
  }
}

template <typename T>
__global__ void k_fill_zero(T* a, long long n) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) a[q] = zero_of(T());
}

// LDS of one k_regular workgroup with `items` (pair, point) items: 18 kernel values and 9 weights
template <bool H>
inline size_t kreg_lds_bytes(int items) {
  return (size_t)items * (18 * sizeof(typename Val<H>::T) + 9 * sizeof(double));
}

// Precalculated-rule pairs (ext_pre: bem_staela3d.f90:592-650, bem_harela3d.f90:628-700) of one
// rule, 64/P pairs per wave: lanes evaluate the kernel at the (pair, point) items into LDS, then each
// lane sums one (pair, kind, c = 3 l + k) row over the rule's points for three element nodes and writes
// it to the pair's 9x3x3 h and g blocks, blocks[162 (blk_base + position) ...].
template <bool H>
__global__ void __launch_bounds__(kWave) k_regular(DevMesh m, const KernelParams* __restrict__ kpp,
                                                   const int* list, int count, int rule,
                                                   typename Val<H>::T* blocks, long long blk_base) {
  typedef typename Val<H>::T T;
  const KernelParams& kp = *kpp;
  const int g = m.ps_gln[rule], P = g * g, B = P >= kWave ? 1 : kWave / P;
  const int base = blockIdx.x * B;
  const int nb = min(B, count - base);
  const int lane = threadIdx.x;
  // LDS sized by the launch for this rule's nb * P items: (pair, point) x (ft[9], fu[9]), then
  // (pair, point) x phi_n J w[9] -- a small rule's workgroup holds less and more of them share a CU
  extern __shared__ double kreg_lds[];
  T* sfs = reinterpret_cast<T*>(kreg_lds);
  double* sw = kreg_lds + (sizeof(T) / sizeof(double)) * 18 * (B * P);
  const int off = m.ps_off[rule];
  for (int it = lane; it < nb * P; it += kWave) {
    int bb = it / P, p = it % P;
    int pid = list[base + bb];
    int e = pid / m.ncp, cp = pid % m.ncp;
    const double* q = m.ps + ((long long)e * m.npts + off + p) * kPsStride;
    double x[3] = {q[0], q[1], q[2]}, n[3] = {q[3], q[4], q[5]};
    double xi[3] = {m.xc[3 * cp], m.xc[3 * cp + 1], m.xc[3 * cp + 2]};
    ext_kernel_row(kp, x, n, xi, &sfs[it * 18]);
    for (int c = 0; c < 9; c++) sw[it * 9 + c] = q[6 + c];
  }
  __syncthreads();
  // one lane per (pair, kind, c = 3 l + k, three element nodes): sums over the rule's points, each
  // kernel value read once and used for the three nodes
  for (int it = lane; it < nb * 54; it += kWave) {
    const int bb = it / 54, o = it % 54, kind = o / 27, c = (o % 27) / 3, n0 = 3 * (o % 3);
    const T* f = &sfs[bb * P * 18 + kind * 9 + c];
    const double* wq = &sw[bb * P * 9 + n0];
    T acc[3] = {zero_of(T()), zero_of(T()), zero_of(T())};
    for (int p = 0; p < P; p++) {
      const T fv = f[p * 18];
      acc[0] += fv * wq[p * 9];
      acc[1] += fv * wq[p * 9 + 1];
      acc[2] += fv * wq[p * 9 + 2];
    }
    const int il = c / 3, ik = c % 3;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const T v = kind ? scale_g(kp, acc[q]) : scale_h(kp, acc[q]);
      blocks[162LL * (blk_base + base + bb) + 81 * kind + n0 + q + 9 * il + 27 * ik] = v;
    }
  }
}

// kernel constants through the constant address space (scalar loads)
typedef const __attribute__((address_space(4))) KernelParams* ConstKP;

// Exterior kernel values at one point, handed to f(l, k, ft) for the nine components of t* and to
// g(c, fu), c = 0..5 for (0,0) (0,1) (0,2) (1,1) (1,2) (2,2), of the symmetric u* (before the
// constants; the values of ext_kernel_row).
template <bool F, bool G, class EmitF, class EmitG>
__device__ inline void ext_point(ConstKP k, const double* x, const double* n,
                                 const double* x_i, double, EmitF&& f, EmitG&& g) {
  const double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  const double s = rsqrt(dot3(rv, rv));
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s};
  if (F) {
    const double s2 = s * s, a = 3.0 * s2 * dot3(dr, n), c = s2 * k->ctet2;
    const double d = c * dot3(dr, n);
    const double cn[3] = {c * n[0], c * n[1], c * n[2]}, ad[3] = {a * dr[0], a * dr[1], a * dr[2]};
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int q = 0; q < 3; q++) {
        double v = ad[l] * dr[q];
        if (l == q) v += d;
        else v += cn[l] * dr[q] - cn[q] * dr[l];
        f(3 * l + q, v);
      }
  }
  if (G) {
    const double a = s * k->cteu2, sd[3] = {s * dr[0], s * dr[1], s * dr[2]};
    int c = 0;
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
      for (int q = l; q < 3; q++) g(c++, l == q ? a + sd[l] * dr[q] : sd[l] * dr[q]);
  }
}

template <bool F, bool G, class EmitF, class EmitG>
__device__ inline void ext_point(ConstKP k, const double* x, const double* n,
                                 const double* x_i, zd, EmitF&& f, EmitG&& g) {
  const double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  double r, s;
  dist_and_inverse(dot3(rv, rv), r, s);
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s};
  zd psi, chi, TT1, TT2, TT3;
  har_factors<F, G>(&k->h, r, s, true, psi, chi, TT1, TT2, TT3);
  if (F) {
    const double drdn = dot3(dr, n);
    const zd a = TT1 * drdn, d = TT2 * drdn;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      // row l: dr_k (a dr_l + TT2 n_l) + n_k (TT3 dr_l) + d delta
      const zd u = a * dr[l] + TT2 * n[l], w = TT3 * dr[l];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        zd v = u * dr[q] + w * n[q];
        if (l == q) v += d;
        f(3 * l + q, v);
      }
    }
  }
  if (G) {
    int c = 0;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const zd u = -(chi * dr[l]);
#pragma unroll
      for (int q = l; q < 3; q++) g(c++, l == q ? psi + u * dr[q] : u * dr[q]);
    }
  }
}

__device__ constexpr int kSym[9] = {0, 1, 2, 1, 3, 4, 2, 4, 5};

// a wave's own LDS stores are seen by its lanes
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sums over the points of one rule of one element for 16 collocation points, one wave, on the FP64
// matrix cores (v_mfma_f64_4x4x4_4b).  A lane evaluates the kernel of pair lane % 16 at point
// p0 + lane / 16: its values are, as they stand, the 16 x 4 left operand, and the weights
// phi_n J w of the four points the 4 x 4 right operands (nodes 0..3, 4..7, 8), so no value goes
// through LDS and no barrier is met.  Per value three of them (48 cycles of the FP64 pipe per SIMD,
// which vector FP64 shares) stand for nine FMAs (36) and the LDS store and loads that those need.
// Result layout: lane holds pair 4 ((lane / 4) % 4) + lane / 16, node 4 m + lane % 4.
// pe: the rule's first point record of the element.
template <bool H, int KIND>
struct TileAcc {
  static constexpr int RC = H ? 2 : 1;
  static constexpr int NF = KIND & kNeedH ? 9 * RC : 1, NG = KIND & kNeedG ? 6 * RC : 1;
  double f[NF][3], g[NG][3];
  __device__ inline void clear() {
#pragma unroll
    for (int c = 0; c < NF; c++) f[c][0] = f[c][1] = f[c][2] = 0.0;
#pragma unroll
    for (int c = 0; c < NG; c++) g[c][0] = g[c][1] = g[c][2] = 0.0;
  }
};
__device__ inline double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ inline void mfma_row(double v, const double* w, double (*acc)[3], int c) {
#pragma unroll
  for (int m = 0; m < 3; m++) acc[c][m] = mfma4(v, w[m], acc[c][m]);
}
__device__ inline void mfma_row(zd v, const double* w, double (*acc)[3], int c) {
#pragma unroll
  for (int m = 0; m < 3; m++) {
    acc[2 * c][m] = mfma4(v.re, w[m], acc[2 * c][m]);
    acc[2 * c + 1][m] = mfma4(v.im, w[m], acc[2 * c + 1][m]);
  }
}

template <bool H, int KIND>
__device__ inline void tile_points(ConstKP kp, const double* __restrict__ pe, int P,
                                   const double* xi, int lane, TileAcc<H, KIND>& acc) {
  typedef typename Val<H>::T T;
  const int k = lane >> 4, j = lane & 3;
  for (int p0 = 0; p0 < P; p0 += 4) {
    // past the last point: the first point's values with zero weights
    const bool in = p0 + k < P;
    const double* q = pe + (in ? p0 + k : 0) * kPsStride;
    const double x[3] = {q[0], q[1], q[2]}, nv[3] = {q[3], q[4], q[5]};
    const double w[3] = {in ? q[6 + j] : 0.0, in ? q[10 + j] : 0.0, in && j == 0 ? q[14] : 0.0};
    ext_point<(KIND & kNeedH) != 0, (KIND & kNeedG) != 0>(
        kp, x, nv, xi, T(), [&](int c, T v) { mfma_row(v, w, acc.f, c); },
        [&](int c, T v) { mfma_row(v, w, acc.g, c); });
  }
}

__device__ inline double tile_value(const double (*a)[3], int c, int m, double) { return a[c][m]; }
__device__ inline zd tile_value(const double (*a)[3], int c, int m, zd) {
  return mkz(a[2 * c][m], a[2 * c + 1][m]);
}

template <typename T>
__device__ inline T lane_xor_add(T v, int mask);
template <>
__device__ inline double lane_xor_add(double v, int mask) { return v + __shfl_xor(v, mask); }
template <>
__device__ inline zd lane_xor_add(zd v, int mask) {
  return mkz(v.re + __shfl_xor(v.re, mask), v.im + __shfl_xor(v.im, mask));
}

// Launches of fewer tiles spread them one by one (runs would leave XCDs without work at the end).
// Runs of 32 keep a rule's neighbouring rows in one L2: 139 us against 188 for the stores alone of a
// launch over 26 x 26 elements.  One eighth of the tiles to each XCD: 847 us against 685, the long
// rules come first and two XCDs take them all.
constexpr int kRunTiles = 16384;

// Columns of four nodes for a tile's 48 rows, on their way to A.
template <typename T>
struct TileLds {
  T v[12][3 * kTileP + 1];
};
typedef const __attribute__((address_space(4))) int* ConstInt;

// where tiles store: A, and the extra points' rows (column stride 3 nx)
template <typename T>
struct TileOut {
  T* A;
  long long lda;
  T* b;
  T* X;
};

// One kind of values (KIND: kNeedH or kNeedG) of a tile: h goes to the columns of unknown u, -g to
// those of unknown t, so the two kinds of an element that needs both store different columns.
template <bool H, int KIND>
__device__ inline void tile_body(const DevMesh& m, const KernelParams& kp,
                                 const int* __restrict__ list, int4 tile, bool twice,
                                 TileLds<typename Val<H>::T>& lds,
                                 const TileOut<typename Val<H>::T>& out) {
  typedef typename Val<H>::T T;
  constexpr bool kH = KIND == kNeedH;
  const int cnt = tile.y, rule = tile.z, e = tile.w, lane = threadIdx.x;
  const int P = m.ps_gln[rule] * m.ps_gln[rule], first = e * m.ncp;
  const double* pe = m.ps + ((long long)e * m.npts + m.ps_off[rule]) * kPsStride;
  // a slot past the tile's pairs repeats the first one; its rows of the result are not stored
  const int slot = lane & 15, cpi = list[tile.x + (slot < cnt ? slot : 0)] - first;
  const double xi[3] = {m.xc[3 * cpi], m.xc[3 * cpi + 1], m.xc[3 * cpi + 2]};
  // lane = row of the tile: three rows per pair
  const int cpr = list[tile.x + (lane < 3 * cnt ? lane / 3 : 0)] - first;
  const int xr = m.cx[cpr];
  T* const arow = (xr < 0 ? out.A + 3LL * m.crow[cpr] : out.X + 3LL * xr) + lane % 3;
  const long long ld = xr < 0 ? out.lda : 3LL * m.nx;
  const bool live = lane < 3 * cnt;
  int code[9];
#pragma unroll
  for (int k = 0; k < 9; k++) code[k] = ((ConstInt)(m.enode + 9LL * e))[k];
  const int fixed = ((ConstInt)(m.emask + e))[0], value = ((ConstInt)(m.emask + e))[1];
  const int to_a = kH ? ~fixed : fixed, to_b = (kH ? fixed : ~fixed) & value;
  TileAcc<H, KIND> acc;
  acc.clear();
  tile_points<H, KIND>((ConstKP)&kp, pe, P, xi, lane, acc);
  const int po = 4 * ((lane >> 2) & 3) + (lane >> 4), j = lane & 3;
  // the lane's value for row component il, node group q, direction ik
  auto val = [&](int il, int ik, int q) {
    if constexpr (kH) return scale_h(kp, tile_value(acc.f, 3 * il + ik, q, T()));
    else return -scale_g(kp, tile_value(acc.g, kSym[3 * il + ik], q, T()));
  };
  constexpr int kNodes[3] = {4, 4, 1};
  // what the columns hold already (nodes that an earlier colour stored): all loads are on their way
  // before the first is waited for
  T w[27];
#pragma unroll
  for (int c = 0; c < 27; c++) {
    w[c] = zero_of(T());
    if (code[c / 3] < 0 && (to_a >> c & 1) && live) w[c] = arow[ld * (3LL * ~code[c / 3] + c % 3)];
  }
#pragma unroll
  for (int q = 0; q < 3; q++) {
    wave_lds_fence();
    if (j < kNodes[q]) {
#pragma unroll
      for (int ik = 0; ik < 3; ik++)
#pragma unroll
        for (int il = 0; il < 3; il++) lds.v[3 * j + ik][3 * po + il] = val(il, ik, q);
    }
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < 3 * kNodes[q]; i++) {
      const int c = 12 * q + i, node = code[c / 3] < 0 ? ~code[c / 3] : code[c / 3];
      if (!(to_a >> c & 1) || !live) continue;
      T* a = arow + ld * (3LL * node + c % 3);
      const T v = lds.v[i][lane];
      if (!twice) *a = w[c] + v;
      else atomic_add(a, v);
    }
  }
  if (to_b & 0x7ffffff) {
    T bs[3] = {zero_of(T()), zero_of(T()), zero_of(T())};
#pragma unroll
    for (int q = 0; q < 3; q++) {
      if (j >= kNodes[q]) continue;
      const int col0 = 3 * m.conn[9 * e + 4 * q + j];
#pragma unroll
      for (int ik = 0; ik < 3; ik++) {
        if (!(to_b >> (3 * (4 * q + j) + ik) & 1)) continue;
        const int col = col0 + ik;
        const double f = m.ctype[col] == 10 ? m.cval[col] * m.nfn[col] : m.cval[col];
#pragma unroll
        for (int il = 0; il < 3; il++) bs[il] = bs[il] - val(il, ik, q) * f;
      }
    }
    const int cp = list[tile.x + (po < cnt ? po : 0)] - first;
    const long long row = 3LL * m.crow[cp];
#pragma unroll
    for (int il = 0; il < 3; il++) {
      bs[il] = lane_xor_add(lane_xor_add(bs[il], 1), 2);
      if (po < cnt && j == 0) atomic_add(&out.b[row + il], bs[il]);
    }
  }
}

// Precalculated-rule pairs scattered into A and b (ext_pre: bem_staela3d.f90:592-650,
// bem_harela3d.f90:628-700; scatter: src/assemble_bem_staela_equation.f90,
// src/assemble_bem_harela_equation.f90), one tile per wave: up to 16 pairs of one element and one
// rule, consecutive entries of the class list (ascending collocation points, so mostly consecutive
// matrix rows).  The tiles of one launch belong to elements of one colour (no shared node) and no two
// points share a row (DevMesh::cx), so no two waves touch the same entry.  The element of the lowest
// colour that holds a node stores its columns, the others add to them: no reset of A and 5 reads
// instead of 9 per element on a structured surface.  The columns go through LDS so that a lane holds
// a row: a store covers 768 consecutive bytes.  t* (tiles h0 .. h0 + n_h) and u* (0 .. n_g) are summed
// by waves of their own, also for elements that need both: together their sums do not fit the
// registers of two waves per SIMD (61 spilled).
// Bound by its FP64 instructions: the 4x4x4 matrix instruction and the vector FMA share one pipe, and
// the sums over the element's nodes are contractions that the former does with a third of the issue
// slots and no LDS traffic for the values.  An open harmonic surface of 26 x 26 elements: 392
// us a launch, 1340 with kernel values staged in LDS by workgroups of 256 and A cleared first; one of
// 50 x 50: 5.0 ms a launch and 13.6 GB, 16.3 ms and 25.8 GB before; a static box of 454 elements 85
// and 157 us.
// One launch over all colours with atomic additions needs no colours, but the chip does 27e9 of them a
// second: 11.8 ms against 4 x 0.695 (26 x 26, this kernel before it stored).
template <bool H>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2)))
    k_regular_tile(DevMesh m, const KernelParams* __restrict__ kpp, const int* __restrict__ list,
                   const int4* __restrict__ tiles, int h0, int n_h, int n_g, int run,
                   TileOut<typename Val<H>::T> out) {
  __shared__ TileLds<typename Val<H>::T> lds;
  // workgroups go to the eight XCDs in turn: `run` consecutive tiles, neighbours in A, to each
  const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
  const int t = ((i / run) * 8 + x) * run + i % run;
  if (t >= n_h + n_g) return;
  const bool is_h = t < n_h;
  const int4 tile = tiles[is_h ? h0 + t : t - n_h];
  const bool twice = m.ekind[tile.w] & kTwice;
  if (is_h) tile_body<H, kNeedH>(m, *kpp, list, tile, twice, lds, out);
  else tile_body<H, kNeedG>(m, *kpp, list, tile, twice, lds, out);
}

// First kernel of an assembly: b := 0, counters (if given) and error flag cleared and, of A and the
// extra rows, what no tile stores: the entries of adaptive and singular pairs (list[0 .. count)) in
// columns that their element would store.  Workgroups: 4 pairs each, then 256 entries of b each.
template <typename T>
__global__ void __launch_bounds__(256) k_begin(DevMesh m, const int* __restrict__ list, int count,
                                               TileOut<T> out, long long* counters, int* err) {
  if (blockIdx.x == 0 && counters) {
    if (threadIdx.x < 2) counters[threadIdx.x] = 0;
    if (threadIdx.x == 0) *err = 0;
  }
  const int pair_blocks = (count + 3) / 4, blk = blockIdx.x;
  if (blk < pair_blocks) {
    const int q = 4 * blk + threadIdx.x / kWave;
    if (q >= count) return;
    const int pid = list[q], e = pid / m.ncp, cp = pid % m.ncp, x = m.cx[cp];
    T* row = x < 0 ? out.A + 3LL * m.crow[cp] : out.X + 3LL * x;
    const long long ld = x < 0 ? out.lda : 3LL * m.nx;
    for (int t = threadIdx.x % kWave; t < 81; t += kWave) {
      const int col = t / 3, node = m.enode[9 * e + col / 3];
      if (node >= 0) row[t % 3 + ld * (3LL * node + col % 3)] = zero_of(T());
    }
    return;
  }
  const int i = 256 * (blk - pair_blocks) + threadIdx.x;
  if (i < 3 * m.nn) out.b[i] = zero_of(T());
}

// rows of the extra points added to their nodes' rows (one thread per component and column of the
// first extra point of a node)
template <typename T>
__global__ void __launch_bounds__(256) k_fold_extra(DevMesh m, TileOut<T> out) {
  const int r = blockIdx.x * 256 + threadIdx.x, x0 = r / 3, il = r % 3;
  if (x0 >= m.nx || (x0 > 0 && m.xnode[x0] == m.xnode[x0 - 1])) return;
  const long long ldx = 3LL * m.nx;
  const int node = m.xnode[x0];
  for (int col = blockIdx.y; col < 3 * m.nn; col += gridDim.y) {
    T v = zero_of(T());
    for (int x = x0; x < m.nx && m.xnode[x] == node; x++) v = v + out.X[3LL * x + il + ldx * col];
    T* a = out.A + 3LL * node + il + out.lda * col;
    *a = *a + v;
  }
}

// ------------------------------------------------------------------------------------------------
// Interior displacements of the precalculated pairs
// ------------------------------------------------------------------------------------------------
// Boundary fields at the precalculated points, with weights and constants: (t, -u) phi J w summed over
// the element's nodes, so that a pair needs 3 products with u* and t* per point instead of their
// 162 integrals over the 9 nodes.
template <typename T>
__global__ void __launch_bounds__(256) k_field(DevMesh m, const KernelParams* __restrict__ kpp,
                                               VecOut<T> vec, T* field) {
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  if (q >= (long long)m.ne * m.npts) return;
  const int e = (int)(q / m.npts);
  const double* w = m.ps + q * kPsStride + 6;
  T f[6];
  for (int c = 0; c < 6; c++) f[c] = zero_of(T());
  for (int n = 0; n < 9; n++) {
    const int sn = m.conn[9 * e + n];
    for (int k = 0; k < 3; k++) {
      f[k] = f[k] + vec.t[3 * sn + k] * w[n];
      f[3 + k] = f[3 + k] - vec.u[3 * sn + k] * w[n];
    }
  }
  for (int k = 0; k < 3; k++) {
    field[6 * q + k] = scale_g(*kpp, f[k]);
    field[6 * q + 3 + k] = scale_h(*kpp, f[3 + k]);
  }
}

// u_l += u*_lk t_k - t*_lk u_k of one point; f: (t, -u) there (the values of ext_point)
__device__ inline void point_values(ConstKP k, const double* rv, const double* n, bool on,
                                    const double* f, double* u) {
  const double s = on ? rsqrt(dot3(rv, rv)) : 0.0;
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s};
  const double rn = dot3(dr, n), s2 = s * s, dt = dot3(dr, f), du = dot3(dr, f + 3), nu = dot3(n, f + 3);
  const double c = s2 * k->ctet2, a = s * dt + 3.0 * s2 * rn * du - c * nu;
  const double ct = s * k->cteu2, cu = c * rn, cn = c * du;
#pragma unroll
  for (int l = 0; l < 3; l++) u[l] += ct * f[l] + cu * f[3 + l] + dr[l] * a + n[l] * cn;
}

__device__ inline void point_values(ConstKP k, const double* rv, const double* n, bool on,
                                    const zd* f, zd* u) {
  double r, s;
  dist_and_inverse(dot3(rv, rv), r, s);
  if (!on) {   // its own r keeps the lane on the branch of its neighbours
    r = r > 0.0 ? r : 1.0;
    s = 0.0;
  }
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s}, rn = dot3(dr, n);
  zd psi, chi, TT1, TT2, TT3;
  har_factors<true, true>(&k->h, r, s, true, psi, chi, TT1, TT2, TT3);
  if (!on) psi = mkz(0.0);   // the other factors meet dr = 0
  const zd dt = f[0] * dr[0] + f[1] * dr[1] + f[2] * dr[2];
  const zd du = f[3] * dr[0] + f[4] * dr[1] + f[5] * dr[2];
  const zd nu = f[3] * n[0] + f[4] * n[1] + f[5] * n[2];
  const zd a = TT1 * (du * rn) + TT3 * nu - chi * dt, cu = TT2 * rn, cn = TT2 * du;
#pragma unroll
  for (int l = 0; l < 3; l++) u[l] += psi * f[l] + cu * f[3 + l] + a * dr[l] + cn * n[l];
}

// One wave per 16 points and `chunk` elements, the sums in registers over the elements.  Four lanes
// share the quadrature points of a pair's own rule, the wave takes as many as the longest of its 16:
// order, the points along a space-filling curve, keeps that close to what each needs, and lanes of one
// rule load one address.  10,000 harmonic points, 216 elements: 0.76 ms; a lane per pair, 64 pairs a
// wave, 1.2 ms; 64 pairs a wave by one rule after the other, its records as scalars, 2.9 ms.
template <bool H>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(3)))
    k_points(DevMesh m, const KernelParams* __restrict__ kpp, const unsigned char* __restrict__ cls,
             const int* __restrict__ order, const typename Val<H>::T* __restrict__ field, int chunk,
             typename Val<H>::T* out) {
  typedef typename Val<H>::T T;
  const ConstKP kp = (ConstKP)kpp;
  const int i = blockIdx.x * 16 + (threadIdx.x & 15), part = threadIdx.x >> 4;
  const bool live = i < m.ncp;
  const int cp = order[live ? i : m.ncp - 1];
  const double xi[3] = {m.xc[3 * cp], m.xc[3 * cp + 1], m.xc[3 * cp + 2]};
  T u[3] = {zero_of(T()), zero_of(T()), zero_of(T())};
  const int e0 = blockIdx.y * chunk, e1 = min(m.ne, e0 + chunk);
  int c = live ? cls[(long long)e0 * m.ncp + cp] : 255;
  for (int e = e0; e < e1; e++) {
    const int next = live ? cls[(long long)min(e + 1, e1 - 1) * m.ncp + cp] : 255;
    const int rule = c < m.n_ps ? c : 0, P = c < m.n_ps ? m.ps_gln[rule] * m.ps_gln[rule] : 0;
    int most = P;
    for (int mask = 1; mask < 16; mask *= 2) most = max(most, __shfl_xor(most, mask));
    const long long q0 = (long long)e * m.npts + m.ps_off[rule];
    for (int p0 = 0; p0 < most; p0 += 4) {
      const int p = p0 + part;
      const long long at = q0 + min(p, max(P - 1, 0));
      const double* q = m.ps + at * kPsStride;
      const double rv[3] = {q[0] - xi[0], q[1] - xi[1], q[2] - xi[2]}, n[3] = {q[3], q[4], q[5]};
      T f[6];
#pragma unroll
      for (int k = 0; k < 6; k++) f[k] = field[6 * at + k];
      point_values(kp, rv, n, p < P, f, u);
    }
    c = next;
  }
  for (int l = 0; l < 3; l++) {
    u[l] = lane_xor_add(lane_xor_add(u[l], 16), 32);
    if (live && part == 0) atomic_add(&out[3 * cp + l], u[l]);
  }
}

// Line integral eps_ijk e_k . t / r over one line3 edge, adaptive Telles + bisection
// (fbem_bem_staela3d_sbie_int_li, bem_staela3d.f90:2245-2376): the 3 independent entries (1,2),
// (1,3), (2,3), by the 16 lanes of a quarter wave.  The lanes walk the bisection together (every
// sub-interval is dyadic: level and index replace a stack) and share the points of a leaf.
__device__ inline void line_integral(const double* Xl, const double* x_i, const QsiParams& q, int ns,
                                     int sub_lane, double* out) {
  const GLTables& G = gl();
  out[0] = out[1] = out[2] = 0;
  int ks = 1, idx = 0;
  for (;;) {
    const double width = 2.0 / (double)(1 << (ks - 1));
    const double xs[2] = {-1.0 + width * idx, -1.0 + width * (idx + 1)};
    double Xs[9];
    if (ks == 1) {
      for (int c = 0; c < 9; c++) Xs[c] = Xl[c];
    } else {
      subdiv_l3(Xl, xs, Xs);
    }
    double cl = length_l3(Xs, 1e-12), bx, rmin, d;
    nearest_l3(Xs, cl, x_i, &bx, &rmin, &d);
    int gln_near = qs_estimate(q, 1, 1, 1, d, &bx);
    if (gln_near == 0 && ks < ns) {
      ks++;
      idx *= 2;
      continue;
    }
    if (gln_near == 0) gln_near = 30;
    const int gln = max(gln_near, 5);
    double tp[4];
    telles11(bx, telles_barr(d), tp);
    for (int kip = sub_lane; kip < gln; kip += 16) {
      double xip, jt;
      telles_xj(tp, G.x11[gln][kip], &xip, &jt);
      double xi = 0.5 * (1.0 - xip) * xs[0] + 0.5 * (1.0 + xip) * xs[1];
      double js = 0.5 * (xs[1] - xs[0]);
      double ph[3], dp[3], x[3] = {0, 0, 0}, T[3] = {0, 0, 0};
      phi_l3(xi, ph);
      dphi_l3(xi, dp);
      for (int kk = 0; kk < 3; kk++)
        for (int c = 0; c < 3; c++) {
          x[c] += ph[kk] * Xl[3 * kk + c];
          T[c] += dp[kk] * Xl[3 * kk + c];
        }
      double jg = sqrt(dot3(T, T));
      double t[3] = {T[0] / jg, T[1] / jg, T[2] / jg};
      double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
      double dr1 = 1.0 / sqrt(dot3(rv, rv));
      double jw = jg * js * jt * G.w11[gln][kip];
      out[0] -= dr1 * t[2] * jw;
      out[1] += dr1 * t[1] * jw;
      out[2] -= dr1 * t[0] * jw;
    }
    // the next interval: out of right halves, then the right half beside
    while (ks > 1 && (idx & 1)) { idx >>= 1; ks--; }
    if (ks == 1) break;
    idx++;
  }
  for (int c = 0; c < 3; c++)
    for (int mask = 1; mask < 16; mask *= 2) out[c] += __shfl_xor(out[c], mask);
}

// local coordinates of the collocation point of a singular pair and, when it is one of the element's
// nodes, that node (else -1)
__device__ inline int singular_xi(const DevMesh& m, const double* X, int e, int cp, double* xi_i) {
  if (m.cel[cp] == e) {
    // an MCA point inside this element: its local coordinates are known exactly
    xi_i[0] = m.cxi[2 * cp];
    xi_i[1] = m.cxi[2 * cp + 1];
  } else {
    double rmin, d;
    const double xc[3] = {m.xc[3 * cp], m.xc[3 * cp + 1], m.xc[3 * cp + 2]};
    nearest_q9(X, m.elem[8 * e], xc, xi_i, &rmin, &d);
  }
  for (int k = 0; k < 9; k++)
    if (xi_i[0] == kXiQ9[k][0] && xi_i[1] == kXiQ9[k][1]) return k;
  return -1;
}

// What a singular pair's integration takes from the geometry alone: where its point lies on the
// element, the polar sub-triangles when that is not a node, and the Stokes line integrals summed over
// the edges that bound an integrated sub-triangle, (1,2), (1,3), (2,3).  Made once, with the lists:
// inside the integration they were four lanes' serial walk, 300 of the 390 us that a launch over a
// small mesh took.  One wave per pair, a quarter wave per edge.
struct SingGeom {
  double hli[3], xi[2], thp[16];
  int node, np, st[8], base[9];   // node: element node at xi or -1; np: quadrature points
};
constexpr int kSingCounts = 64;   // the points are counted in that many places
__global__ void __launch_bounds__(kWave) k_sing_geom(DevMesh m,
                                                     const QsiParams* __restrict__ qsp_li,
                                                     const int* __restrict__ list, SingGeom* geo,
                                                     unsigned long long* np) {
  const int lane = threadIdx.x, edge = lane >> 4;
  const int pid = list[blockIdx.x], e = pid / m.ncp, cp = pid % m.ncp;
  double X[27], xi_i[2], x_i[3], o[3] = {0, 0, 0};
  load_X(m, e, X);
  const int k = singular_xi(m, X, e, cp, xi_i);
  q9_x(X, xi_i[0], xi_i[1], x_i);
  int st[8], nst;
  SingGeom& out = geo[blockIdx.x];
  if (k >= 0) {
    nst = c_polar[k].n;
    for (int s = 0; s < nst; s++) st[s] = c_polar[k].st[s];
    if (lane == 0) out.np = c_polar_np[k];
  } else {
    double th[16], thp[16];
    nst = polar_setup_q(xi_i, st, th, thp);
    if (lane == 0) {
      int base = 0;
      for (int s = 0; s < 8; s++) {
        out.base[s] = base;
        if (s < nst) {
          base += 15 * (5 + (int)round(25.0 * (th[2 * s + 1] - th[2 * s]) / kPi_2));
          out.st[s] = st[s];
          out.thp[2 * s] = thp[2 * s];
          out.thp[2 * s + 1] = thp[2 * s + 1];
        }
      }
      out.base[8] = base;
      out.np = base;
    }
  }
  bool integrate = false;
  for (int s = 0; s < nst; s++)
    if (st[s] == 2 * edge + 1 || st[s] == 2 * edge + 2) integrate = true;
  if (integrate) {
    double Xl[9];
    for (int j = 0; j < 3; j++)
      for (int c = 0; c < 3; c++) Xl[3 * j + c] = X[3 * kEdgeQ9[edge][j] + c];
    line_integral(Xl, x_i, *qsp_li, 16, lane & 15, o);
  }
  for (int c = 0; c < 3; c++) {
    o[c] += __shfl_xor(o[c], 16);
    o[c] += __shfl_xor(o[c], 32);
  }
  if (lane == 0) {
    for (int c = 0; c < 3; c++) out.hli[c] = o[c];
    out.xi[0] = xi_i[0];
    out.xi[1] = xi_i[1];
    out.node = k;
    atomicAdd(&np[blockIdx.x % kSingCounts], (unsigned long long)out.np);
  }
}

// point (kt, kr) of a sub-triangle's rule at xi_i: local coordinates and rho x weights
__device__ __attribute__((noinline)) void polar_point(const double* xi_i, int st, double thp0, double thp1, int nt,
                                   int kt, int kr, double* xi, double* w) {
  const GLTables& G = gl();
  const double jtp = thp1 - thp0, tpv = jtp * G.x01[nt][kt] + thp0;
  double theta, rhoij, sn, cs;
  polar_angular_q(xi_i, st, tpv, &theta, &rhoij);
  sincos(theta, &sn, &cs);
  const double rho = rhoij * G.x01[15][kr];
  xi[0] = xi_i[0] + rho * cs;
  xi[1] = xi_i[1] + rho * sn;
  *w = rho * jtp * G.w01[nt][kt] * G.w01[15][kr];
}

__global__ void k_polar_table() {
  const int k = blockIdx.y, p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= c_polar_np[k]) return;
  const PolarSet& ps = c_polar[k];
  int s = 0, base = 0;
  while (p >= base + ps.ngt[s] * 15) base += 15 * ps.ngt[s++];
  const int q = p - base;
  polar_point(kXiQ9[k], ps.st[s], ps.thp[2 * s], ps.thp[2 * s + 1], ps.ngt[s], q / 15, q % 15,
              g_polar_pts[k][p], &g_polar_pts[k][p][2]);
}

// Kernel values of the singular integration (bem_staela3d.f90:1303-1322; bem_harela3d.f90:
// 1418-1438), h += ft*phi*jw + fc*(phi-phi_i)*jw, g += fu*phi*jw, as rows of real numbers: ft first
// (static: the 6 of a symmetric 3 x 3, harmonic: 9 complex), then the 6 of the symmetric fu, from
// row fc0 on the 3 of the antisymmetric fc without its constant factor (ctet2, lead of TT2).
template <bool H, int KIND>
struct SingRows {
  static constexpr int NH = KIND & kNeedH ? (H ? 18 : 6) : 0, NG = KIND & kNeedG ? (H ? 12 : 6) : 0;
  static constexpr int fc0 = (NH + NG + 3) / 4 * 4;                // rows in groups of four
  static constexpr int NR = fc0 + (KIND & kNeedH ? 4 : 0);
};

template <int KIND>
__device__ inline void sing_rows(ConstKP k, const double* x, const double* n, const double* x_i,
                                 double* v, double) {
  typedef SingRows<false, KIND> R;
  const double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  const double s = rsqrt(dot3(rv, rv)), s2 = s * s;
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s}, drdn = dot3(dr, n);
  const double a = s2 * drdn, ac = a * k->ctet2, u = s * k->cteu2;
  int c = 0;
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int q = l; q < 3; q++, c++) {
      const double rr = dr[l] * dr[q];
      if (KIND & kNeedH) v[c] = 3.0 * a * rr + (l == q ? ac : 0.0);
      if (KIND & kNeedG) v[R::NH + c] = s * rr + (l == q ? u : 0.0);
    }
  if (KIND & kNeedH) {
    v[R::fc0] = s2 * (n[0] * dr[1] - n[1] * dr[0]);
    v[R::fc0 + 1] = s2 * (n[0] * dr[2] - n[2] * dr[0]);
    v[R::fc0 + 2] = s2 * (n[1] * dr[2] - n[2] * dr[1]);
  }
}

template <int KIND>
__device__ inline void sing_rows(ConstKP k, const double* x, const double* n, const double* x_i,
                                 double* v, zd) {
  typedef SingRows<true, KIND> R;
  const double rv[3] = {x[0] - x_i[0], x[1] - x_i[1], x[2] - x_i[2]};
  double r, s;
  dist_and_inverse(dot3(rv, rv), r, s);
  const double dr[3] = {rv[0] * s, rv[1] * s, rv[2] * s}, drdn = dot3(dr, n), s2 = s * s;
  zd psi, chi, TT1, TT2, TT3;
  har_factors<(KIND & kNeedH) != 0, (KIND & kNeedG) != 0>(&k->h, r, s, false, psi, chi, TT1, TT2, TT3);
  if (KIND & kNeedH) {
    const zd a = (TT1 + mkz(k->h.lead[2][0], k->h.lead[2][1]) * s2) * drdn;
    const zd d = (TT2 + mkz(k->h.lead[3][0], k->h.lead[3][1]) * s2) * drdn;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const zd u = a * dr[l] + TT2 * n[l], w = TT3 * dr[l];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        zd f = u * dr[q] + w * n[q];
        if (l == q) f += d;
        v[2 * (3 * l + q)] = f.re;
        v[2 * (3 * l + q) + 1] = f.im;
      }
    }
    v[R::fc0] = s2 * (n[0] * dr[1] - n[1] * dr[0]);
    v[R::fc0 + 1] = s2 * (n[0] * dr[2] - n[2] * dr[0]);
    v[R::fc0 + 2] = s2 * (n[1] * dr[2] - n[2] * dr[1]);
  }
  if (KIND & kNeedG) {
    int c = 0;
#pragma unroll
    for (int l = 0; l < 3; l++) {
      const zd u = -(chi * dr[l]);
#pragma unroll
      for (int q = l; q < 3; q++, c++) {
        const zd f = l == q ? psi + u * dr[q] : u * dr[q];
        v[R::NH + 2 * c] = f.re;
        v[R::NH + 2 * c + 1] = f.im;
      }
    }
  }
}

// LDS of one pair integrated by W waves: 12 rows of kernel values and phi, jw of a wave's 64 points
// (rows 72 doubles apart: the matrix operands' loads meet no bank twice), then the waves' sums.
constexpr int kRowStride = 72, kPassRows = 12;
template <int W>
struct PairLds {
  union {
    struct {
      double f[W][kPassRows][kRowStride];
      double ph[W][10][kRowStride];
    };
    double sum[W][36][9];
  };
};

// acc[g][q] += sum over the wave's 64 points of (rows 4 g .. 4 g + 3) x (weights of nodes 4 q ..
// 4 q + 3): the lane's values v of its point go through LDS, 12 rows at a time, into the layout of
// the left operand; each of the four blocks of an instruction takes four of 16 points, so the result
// is summed over lane bits 2, 3 at the end (rows_reduce).  From row FC on the weights are
// (phi - phi_i) jw.  A point without weight carries jw = 0 and finite values.
template <int NR, int FC>
__device__ inline void rows_mfma(const double* v, const double* ph, double jw, const double* pf_i,
                                 double (*f)[kRowStride], double (*sp)[kRowStride], int lane,
                                 double (*acc)[3]) {
  wave_lds_fence();
#pragma unroll
  for (int n = 0; n < 9; n++) sp[n][lane] = ph[n];
  sp[9][lane] = jw;
  const int i = lane & 3, at = 4 * (lane >> 4) + ((lane >> 2) & 3);
#pragma unroll
  for (int r0 = 0; r0 < NR; r0 += kPassRows) {
    wave_lds_fence();
#pragma unroll
    for (int r = r0; r < r0 + kPassRows && r < NR; r++) f[r - r0][lane] = v[r];
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const double j = sp[9][16 * t + at], p0 = sp[i][16 * t + at], p1 = sp[4 + i][16 * t + at];
      const double p2 = sp[8][16 * t + at];
#pragma unroll
      for (int r = r0; r < r0 + kPassRows && r < NR; r += 4) {
        const double a = f[r - r0 + i][16 * t + at];
        const bool fc = r >= FC;
        acc[r / 4][0] = mfma4(a, (fc ? p0 - pf_i[0] : p0) * j, acc[r / 4][0]);
        acc[r / 4][1] = mfma4(a, (fc ? p1 - pf_i[1] : p1) * j, acc[r / 4][1]);
        acc[r / 4][2] = mfma4(a, i == 0 ? (fc ? p2 - pf_i[2] : p2) * j : 0.0, acc[r / 4][2]);
      }
    }
  }
}

// sums of the workgroup's W waves (W = 1: of the calling wave alone): lds.sum[0][row][node] afterwards
template <int NR, int W>
__device__ inline void rows_reduce(double (*acc)[3], PairLds<W>& lds, int wave, int lane) {
  if (W > 1) __syncthreads();
  else wave_lds_fence();
#pragma unroll
  for (int g = 0; g < NR / 4; g++)
#pragma unroll
    for (int q = 0; q < 3; q++) {
      double t = acc[g][q];
      t += __shfl_xor(t, 4);
      t += __shfl_xor(t, 8);
      const int n = 4 * q + (lane & 3);
      if (!(lane & 12) && n < 9) lds.sum[wave][4 * g + (lane >> 4)][n] = t;
    }
  if (W > 1) __syncthreads();
  else wave_lds_fence();
  if (W > 1) {
    for (int o = threadIdx.x; o < NR * 9; o += W * kWave) {
      double t = lds.sum[0][0][o];
      for (int w = 1; w < W; w++) t += lds.sum[w][0][o];
      lds.sum[0][0][o] = t;
    }
    __syncthreads();
  }
}

// Output of one pair: value(kind, l, k, n) -> h (0) or g (1) with the kernel constants.  Items
// t < 81 are (n, l, k) each: scatter into A and b (scatter of
// src/assemble_bem_{staela,harela}_equation.f90), the pair's blocks, or the displacement of its point
// (summed over the calling wave's items).
template <bool H, int KIND, class Value>
__device__ inline void pair_output(const DevMesh& m, int e, int cp, int t,
                                   typename Val<H>::T* A, long long lda, typename Val<H>::T* b,
                                   typename Val<H>::T* block, const VecOut<typename Val<H>::T>& vec,
                                   Value&& value) {
  typedef typename Val<H>::T T;
  T part = zero_of(T());
  if (t < 81) {
    const int il = t % 3, n = (t / 3) % 9, ik = t / 27;
    const int sn = m.conn[9 * e + n];
    const long long col = 3LL * sn + ik;
    if (block) {
      const int o = n + 9 * il + 27 * ik;
      block[o] = value(0, il, ik, n);
      block[81 + o] = value(1, il, ik, n);
    } else if (vec.out) {
      part = value(1, il, ik, n) * vec.t[col] - value(0, il, ik, n) * vec.u[col];
    } else {
      const long long row = 3LL * m.crow[cp] + il;
      const int ct = m.ctype[col];
      const double cv = m.cval[col];
      atomic_add(&A[row + lda * col], ct == 0 ? -value(1, il, ik, n) : value(0, il, ik, n));
      if (KIND == (kNeedH | kNeedG) && cv != 0.0) {
        if (ct == 0) atomic_add(&b[row], value(0, il, ik, n) * -cv);
        else atomic_add(&b[row], value(1, il, ik, n) * (ct == 1 ? cv : cv * m.nfn[col]));
      }
    }
  }
  if (vec.out) {
    for (int il = 0; il < 3; il++) {
      T q = t < 81 && t % 3 == il ? part : zero_of(T());
      for (int mask = 1; mask < kWave; mask *= 2) q = lane_xor_add(q, mask);
      if (t % kWave == 0 && t < 81) atomic_add(&vec.out[3 * cp + il], q);
    }
  }
}

// Singular pairs: fbem_bem_staela3d_sbie_int (bem_staela3d.f90:1100-1381) and
// fbem_bem_harela3d_sbie_int (bem_harela3d.f90:1174-1472).  A pair's points are spread over four waves
// and the rows summed over them by the FP64 matrix cores, which leaves a lane's share of the sums in
// registers: as one wave per pair with tables and line integrals made inside, a launch of its own took
// 391 us on a cube of 24 static elements (23 now), 550 on a sphere of 96 (69), 2112 on an open surface
// of 26 x 26 (351).
constexpr int kSingWaves = 4;
template <bool H, int KIND>
__device__ inline void singular_body(const DevMesh& m, ConstKP kp, int e, int cp,
                                     const SingGeom* __restrict__ geo, PairLds<kSingWaves>& lds,
                                     typename Val<H>::T* A, long long lda, typename Val<H>::T* b,
                                     typename Val<H>::T* block,
                                     const VecOut<typename Val<H>::T>& vec) {
  typedef typename Val<H>::T T;
  typedef SingRows<H, KIND> R;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  double X[27], x_i[3], pf[9];
  load_X(m, e, X);
  const double xi_i[2] = {geo->xi[0], geo->xi[1]};
  const int node = geo->node, P = geo->np;
  q9_x(X, xi_i[0], xi_i[1], x_i);
  phi_q9(xi_i[0], xi_i[1], pf);
  double acc[R::NR / 4][3];
#pragma unroll
  for (int g = 0; g < R::NR / 4; g++) acc[g][0] = acc[g][1] = acc[g][2] = 0.0;
  const int i = lane & 3;
  const double pfi[3] = {pf[i], pf[4 + i], pf[8]};
  for (int start = wave * kWave; start < P; start += kSingWaves * kWave) {
    const int p = min(start + lane, P - 1);
    double xi[2], w;
    if (node >= 0) {
      const double* q = g_polar_pts[node][p];
      xi[0] = q[0];
      xi[1] = q[1];
      w = q[2];
    } else {
      int s = 0;
      while (p >= geo->base[s + 1]) s++;
      const int q = p - geo->base[s];
      polar_point(xi_i, geo->st[s], geo->thp[2 * s], geo->thp[2 * s + 1],
                  (geo->base[s + 1] - geo->base[s]) / 15, q / 15, q % 15, xi, &w);
    }
    double x[3], T1[3], T2[3], N[3], ph[9], v[R::NR];
    q9_geom(X, xi[0], xi[1], x, T1, T2);
    cross3(T1, T2, N);
    const double jg = sqrt(dot3(N, N)), ij = 1.0 / jg;
    const double n[3] = {N[0] * ij, N[1] * ij, N[2] * ij};
    phi_q9(xi[0], xi[1], ph);
#pragma unroll
    for (int r = 0; r < R::NR; r++) v[r] = 0.0;
    sing_rows<KIND>(kp, x, n, x_i, v, T());
    rows_mfma<R::NR, (KIND & kNeedH) ? R::fc0 : R::NR>(
        v, ph, start + lane < P ? jg * w : 0.0, pfi, lds.f[wave], lds.ph[wave], lane, acc);
  }
  rows_reduce<R::NR, kSingWaves>(acc, lds, wave, lane);
  const double(*S)[9] = lds.sum[0];
  pair_output<H, KIND>(
      m, e, cp, (int)threadIdx.x, A, lda, b, block, vec, [&](int kind, int il, int ik, int n) {
        const int c = il == ik ? -1 : il + ik - 1;   // (0,1) 0, (0,2) 1, (1,2) 2
        if constexpr (H) {
          const int r = kind ? R::NH + 2 * kSym[3 * il + ik] : 2 * (3 * il + ik);
          T v = mkz(S[r][n], S[r + 1][n]);
          if (kind) return mkz(kp->h.cte_u[0], kp->h.cte_u[1]) * v;
          if (c >= 0) {
            const double a = S[R::fc0 + c][n] + pf[n] * geo->hli[c];
            v += mkz(kp->h.lead[3][0], kp->h.lead[3][1]) * (il < ik ? a : -a);
          }
          return mkz(kp->h.cte_t[0], kp->h.cte_t[1]) * v;
        } else {
          double v = S[(kind ? R::NH : 0) + kSym[3 * il + ik]][n];
          if (kind) return v * kp->cteu1;
          if (c >= 0) {
            const double a = S[R::fc0 + c][n] + pf[n] * geo->hli[c];
            v += kp->ctet2 * (il < ik ? a : -a);
          }
          return v * kp->ctet1;
        }
      });
}

// One workgroup of four waves per pair, a wave 64 polar points at a time; per point the values are
// few real rows (the antisymmetric part and u* by their distinct components), summed against the
// nine weights on the FP64 matrix cores.
template <bool H>
__device__ inline void singular_pair(const DevMesh& m, ConstKP kp, int pid,
                                     const SingGeom* __restrict__ geo, PairLds<kSingWaves>& lds,
                                     typename Val<H>::T* A, long long lda, typename Val<H>::T* b,
                                     typename Val<H>::T* block,
                                     const VecOut<typename Val<H>::T>& vec) {
  const int e = pid / m.ncp, cp = pid % m.ncp;
  const int kind = block || vec.out ? kNeedH | kNeedG : m.ekind[e] & (kNeedH | kNeedG);
  if (kind == kNeedH) singular_body<H, kNeedH>(m, kp, e, cp, geo, lds, A, lda, b, block, vec);
  else if (kind == kNeedG) singular_body<H, kNeedG>(m, kp, e, cp, geo, lds, A, lda, b, block, vec);
  else singular_body<H, kNeedH | kNeedG>(m, kp, e, cp, geo, lds, A, lda, b, block, vec);
}

// Adaptive quasi-singular pairs: fbem_bem_staela3d_sbie_ext_adp (bem_staela3d.f90:973-1096,
// bem_harela3d.f90:1050-1172) with ext_st leaves (:654-969, :702-1048).
//
// Root of a pair's subdivision tree: nearest point and rule order of the whole element, gln = 0 where
// it is to be subdivided.  96 % of the pairs are a single leaf: the search, a serial chain of double-
// double Newton steps, is taken by four lanes per pair in a kernel of its own, 16 pairs a wave, when
// the lists are made (a wave of the integration ran it in one lane).
struct AdaptGeom {
  double barxi[2], d;
  int gln, pad;
};

// order of the sub-element (nodes X, size cl) at tree level ks, 0: subdivide
__device__ inline int leaf_order(const QsiParams& qsp, const double* X, double cl,
                                 const double* x_i, int ks, int ns_max, double* barxi, double* d) {
  double rmin;
  nearest_q9_wave<true>(true, X, cl, x_i, barxi, &rmin, d);
  const int gln = qs_estimate(qsp, 1, 2, 5, *d, barxi);
  return gln == 0 && ks == ns_max ? 30 : gln;
}

// Records of `count` listed pairs in one buffer; behind them what is to be subdivided and what the
// others, single leaves, hold.
struct AdaptSum {
  unsigned long long points;   // quadrature points and number of the single leaves
  int leaves, n_tree;          // pairs to be subdivided
  __host__ __device__ int* tree() { return (int*)(this + 1); }   // their list positions
};
__host__ __device__ inline size_t adapt_geom_bytes(size_t count) {
  return count * (sizeof(AdaptGeom) + sizeof(int)) + sizeof(AdaptSum);
}
__host__ __device__ inline AdaptSum* adapt_sum(AdaptGeom* geo, size_t count) {
  return (AdaptSum*)(geo + count);
}

__global__ void __launch_bounds__(kWave) k_adapt_geom(DevMesh m, const QsiParams* __restrict__ qsp,
                                                      const int* __restrict__ list, int count,
                                                      AdaptGeom* geo) {
  const int q = blockIdx.x * 16 + (threadIdx.x >> 2), sub = threadIdx.x & 3;
  const int pid = list[min(q, count - 1)], e = pid / m.ncp, cp = pid % m.ncp;
  double X[27], barxi[2], d;
  load_X(m, e, X);
  const double x_i[3] = {m.xc[3 * cp], m.xc[3 * cp + 1], m.xc[3 * cp + 2]};
  const int gln = leaf_order(*qsp, X, m.elem[8 * e], x_i, 1, m.ns_max, barxi, &d);
  AdaptSum* sum = adapt_sum(geo, count);
  const bool mine = q < count && sub == 0;
  const int order = gln ? max(gln, (int)m.elem[8 * e + 5]) : 0;
  if (mine) {
    AdaptGeom& g = geo[q];
    g.barxi[0] = barxi[0];
    g.barxi[1] = barxi[1];
    g.d = d;
    g.gln = order;
    g.pad = 0;
    if (gln == 0) sum->tree()[atomicAdd(&sum->n_tree, 1)] = q;
  }
  int points = mine ? order * order : 0;
  for (int mask = 4; mask < kWave; mask *= 2) points += __shfl_xor(points, mask);
  const int leaves = __popcll(__ballot(mine && order));
  if (threadIdx.x == 0) {
    atomicAdd(&sum->points, (unsigned long long)points);
    atomicAdd(&sum->leaves, leaves);
  }
}

// A leaf: the square of centre c and half width h, the nearest point in its own coordinates.
struct Leaf {
  double c[2], h, barxi[2], d;
  int gln, pad;
};
constexpr int kLeaves = 32, kWalkWidth = 8;
// The walk takes the kWalkWidth topmost sub-elements of its stack at a time and puts the parts of those
// that it splits, at most 4 kWalkWidth, in their place.  Of the parts that one step has put there, at most
// 3 kWalkWidth are left below those of a later step, and the shallowest level that a step puts there is
// deeper than what the step below put: there are fewer than kMaxNs steps' parts.  (Simulated with random
// splits to level 20: 408 entries at most; with everything split to level 9: 160.)
constexpr int kWalkStack = 3 * kWalkWidth * kMaxNs + 4 * kWalkWidth;
struct WalkLds {
  unsigned long long stk[kWalkStack];   // level << 48 | ix << 24 | iy of the 2^(level-1) grid
  Leaf leaf[kLeaves];
};

// One step of the walk: the topmost sub-elements of the stack (a team of four lanes each) become
// leaves or are replaced by their four parts.  sp, nl: entries on the stack, leaves.
__device__ __attribute__((noinline)) void walk_step(const QsiParams& qsp, const double* X,
                                                    const double* x_i, int ns_max, int gln_far,
                                                    WalkLds& w, int& sp, int& nl) {
  const int lane = threadIdx.x % kWave, team = lane >> 2, sub = lane & 3;
  const int n = min(sp, kWalkWidth);
  const unsigned long long node = w.stk[sp - 1 - min(team, n - 1)];
  const int ks = (int)(node >> 48), ix = (int)(node >> 24) & 0xffffff, iy = (int)node & 0xffffff;
  const double width = 2.0 / (double)(1 << (ks - 1));
  const double a0 = -1.0 + width * ix, b0 = -1.0 + width * iy, a1 = a0 + width, b1 = b0 + width;
  const double xs[8] = {a0, b0, a1, b0, a1, b1, a0, b1};
  double Xs[27], barxi[2], d;
  subdiv_q9(X, xs, Xs);
  const double cl = clen_q9_team(Xs, 1e-12, sub);
  const int gln = leaf_order(qsp, Xs, cl, x_i, ks, ns_max, barxi, &d);
  const bool mine = team < n && sub == 0;
  const unsigned long long split = __ballot(mine && gln == 0), leaf = __ballot(mine && gln != 0);
  const unsigned long long below = (1ull << lane) - 1ull;
  wave_lds_fence();   // the step's stack entries are read
  if (mine && gln == 0) {
    unsigned long long* t = w.stk + (sp - n) + 4 * __popcll(split & below);
    const unsigned long long up = (unsigned long long)(ks + 1) << 48;
    for (int c = 0; c < 4; c++)
      t[c] = up | (unsigned long long)(2 * ix + (c == 1 || c == 2)) << 24 |
             (unsigned long long)(2 * iy + (c >= 2));
  } else if (mine) {
    Leaf& l = w.leaf[nl + __popcll(leaf & below)];
    l.c[0] = 0.5 * (a0 + a1);
    l.c[1] = 0.5 * (b0 + b1);
    l.h = 0.5 * width;
    l.barxi[0] = barxi[0];
    l.barxi[1] = barxi[1];
    l.d = d;
    l.gln = max(gln, gln_far);
  }
  wave_lds_fence();
  sp += 4 * __popcll(split) - n;
  nl += __popcll(leaf);
}

template <bool H, int KIND>
struct ExtRows {
  static constexpr int RC = H ? 2 : 1;
  static constexpr int NH = KIND & kNeedH ? 9 * RC : 0, NG = KIND & kNeedG ? 6 * RC : 0;
  static constexpr int NR = (NH + NG + 3) / 4 * 4;
};
__device__ inline void put_row(double* v, int c, double x) { v[c] = x; }
__device__ inline void put_row(double* v, int c, zd x) {
  v[2 * c] = x.re;
  v[2 * c + 1] = x.im;
}

// sums of one leaf: Telles rule of order gln on the square (c, h)
template <bool H, int KIND>
__device__ inline int leaf_sums(ConstKP kp, const double* X, const double* x_i, const double* c,
                                double h, const double* barxi, double d, int gln,
                                PairLds<1>& lds, int lane, double (*acc)[3]) {
  typedef typename Val<H>::T T;
  typedef ExtRows<H, KIND> R;
  const GLTables& G = gl();
  double tp1[4], tp2[4];
  const double barr = telles_barr(d);
  telles11(barxi[0], barr, tp1);
  telles11(barxi[1], barr, tp2);
  const int P = gln * gln;
  for (int start = 0; start < P; start += kWave) {
    const int p = min(start + lane, P - 1), k1 = p / gln, k2 = p % gln;
    double xp0, xp1, jt1, jt2;
    telles_xj(tp1, G.x11[gln][k1], &xp0, &jt1);
    telles_xj(tp2, G.x11[gln][k2], &xp1, &jt2);
    const double xi0 = c[0] + h * xp0, xi1 = c[1] + h * xp1;
    double x[3], T1[3], T2[3], N[3], ph[9], v[R::NR];
    q9_geom(X, xi0, xi1, x, T1, T2);
    cross3(T1, T2, N);
    const double jg = sqrt(dot3(N, N)), ij = 1.0 / jg;
    const double n[3] = {N[0] * ij, N[1] * ij, N[2] * ij};
    const double jw = jg * (h * h) * (jt1 * jt2) * (G.w11[gln][k1] * G.w11[gln][k2]);
    phi_q9(xi0, xi1, ph);
#pragma unroll
    for (int r = R::NH + R::NG; r < R::NR; r++) v[r] = 0.0;
    ext_point<(KIND & kNeedH) != 0, (KIND & kNeedG) != 0>(
        kp, x, n, x_i, T(), [&](int q, T f) { put_row(v, q, f); },
        [&](int q, T f) { put_row(v + R::NH, q, f); });
    rows_mfma<R::NR, R::NR>(v, ph, start + lane < P ? jw : 0.0, nullptr, lds.f[0], lds.ph[0], lane,
                            acc);
  }
  return P;
}

template <bool H, int KIND, bool TREE>
__device__ inline void adaptive_body(const DevMesh& m, const QsiParams& qsp, ConstKP kp, int e,
                                     int cp, const AdaptGeom& root, PairLds<1>& lds, WalkLds* walk,
                                     typename Val<H>::T* A, long long lda, typename Val<H>::T* b,
                                     long long* counters, typename Val<H>::T* block,
                                     const VecOut<typename Val<H>::T>& vec) {
  typedef typename Val<H>::T T;
  typedef ExtRows<H, KIND> R;
  const int lane = threadIdx.x % kWave, gln_far = (int)m.elem[8 * e + 5];
  double X[27];
  load_X(m, e, X);
  const double x_i[3] = {m.xc[3 * cp], m.xc[3 * cp + 1], m.xc[3 * cp + 2]};
  double acc[R::NR / 4][3];
#pragma unroll
  for (int g = 0; g < R::NR / 4; g++) acc[g][0] = acc[g][1] = acc[g][2] = 0.0;
  int leaves = 1, npts = 0;
  if (!TREE) {
    const double c[2] = {0.0, 0.0};
    npts = leaf_sums<H, KIND>(kp, X, x_i, c, 1.0, root.barxi, root.d, root.gln, lds,
                              lane, acc);
  } else {
    int sp = 4, nl = 0;
    if (lane < 4)
      walk->stk[lane] = 2ull << 48 | (unsigned long long)(lane == 1 || lane == 2) << 24 |
                        (unsigned long long)(lane >= 2);
    wave_lds_fence();
    // leaves are integrated in batches; the walk goes on from its stack
    for (leaves = 0;;) {
      while (sp > 0 && nl + kWalkWidth <= kLeaves)
        walk_step(qsp, X, x_i, m.ns_max, gln_far, *walk, sp, nl);
      for (int l = 0; l < nl; l++) {
        const Leaf& q = walk->leaf[l];
        npts += leaf_sums<H, KIND>(kp, X, x_i, q.c, q.h, q.barxi, q.d,
                                   __builtin_amdgcn_readfirstlane(q.gln), lds, lane, acc);
      }
      leaves += nl;
      nl = 0;
      if (sp == 0) break;
      wave_lds_fence();
    }
  }
  rows_reduce<R::NR, 1>(acc, lds, 0, lane);
  const double(*S)[9] = lds.sum[0];
  auto value = [&](int kind, int il, int ik, int n) {
    const int c = kind ? R::NH + R::RC * kSym[3 * il + ik] : R::RC * (3 * il + ik);
    if constexpr (H) {
      const T v = mkz(S[c][n], S[c + 1][n]);
      return kind ? mkz(kp->h.cte_u[0], kp->h.cte_u[1]) * v : mkz(kp->h.cte_t[0], kp->h.cte_t[1]) * v;
    } else {
      return S[c][n] * (kind ? kp->cteu1 : kp->ctet1);
    }
  };
  pair_output<H, KIND>(m, e, cp, lane, A, lda, b, block, vec, value);
  pair_output<H, KIND>(m, e, cp, lane + kWave, A, lda, b, block, vec, value);
  if (TREE && lane == 0) {
    atomicAdd((unsigned long long*)&counters[0], (unsigned long long)npts);
    atomicAdd((unsigned long long*)&counters[1], (unsigned long long)leaves);
  }
}

template <bool H, bool TREE>
__device__ inline void adaptive_pair(const DevMesh& m, const QsiParams* __restrict__ qsp, ConstKP kp,
                                     const int* __restrict__ list,
                                     const AdaptGeom* __restrict__ geo, int q, PairLds<1>& lds,
                                     WalkLds* walk, typename Val<H>::T* A, long long lda,
                                     typename Val<H>::T* b, long long* counters,
                                     typename Val<H>::T* blocks,
                                     const VecOut<typename Val<H>::T>& vec) {
  const int pid = list[q], e = pid / m.ncp, cp = pid % m.ncp;
  typename Val<H>::T* block = blocks ? blocks + 162LL * q : nullptr;
  const int kind = block || vec.out ? kNeedH | kNeedG : m.ekind[e] & (kNeedH | kNeedG);
  if (kind == kNeedH)
    adaptive_body<H, kNeedH, TREE>(m, *qsp, kp, e, cp, geo[q], lds, walk, A, lda, b, counters,
                                   block, vec);
  else if (kind == kNeedG)
    adaptive_body<H, kNeedG, TREE>(m, *qsp, kp, e, cp, geo[q], lds, walk, A, lda, b, counters,
                                   block, vec);
  else
    adaptive_body<H, kNeedH | kNeedG, TREE>(m, *qsp, kp, e, cp, geo[q], lds, walk, A, lda, b,
                                            counters, block, vec);
}

// err[q * nr + r] = max(max|h - h_ref| / max|h_ref|, max|g - g_ref| / max|g_ref|) of pair q
// (one wave per pair; blocks of 162 values, h then g)
template <typename T>
__global__ void __launch_bounds__(kWave) k_block_err(const T* ref, const T* blk, int nr, int r,
                                                     double* err) {
  const long long q = blockIdx.x;
  const int lane = threadIdx.x;
  double dh = 0, mh = 0, dg = 0, mg = 0;
  for (int o = lane; o < 162; o += kWave) {
    const double a = mag(ref[162 * q + o]), dd = mag(blk[162 * q + o] - ref[162 * q + o]);
    if (o < 81) { mh = fmax(mh, a); dh = fmax(dh, dd); }
    else { mg = fmax(mg, a); dg = fmax(dg, dd); }
  }
  for (int off = 32; off > 0; off >>= 1) {
    dh = fmax(dh, __shfl_xor(dh, off));
    mh = fmax(mh, __shfl_xor(mh, off));
    dg = fmax(dg, __shfl_xor(dg, off));
    mg = fmax(mg, __shfl_xor(mg, off));
  }
  if (lane == 0) {
    const double r0 = mag(ref[162 * q]);
    // a reference that is not a number gives a NaN error
    err[q * nr + r] = r0 != r0 ? r0 : fmax(mh > 0 ? dh / mh : dh, mg > 0 ? dg / mg : dg);
  }
}

// label of pair q: class of the cheapest precalculated rule with err <= tau (class = order - 2),
// MFB_QNET_CLASSES - 1 (adaptive) when none is; written to labels[idx[q]]
__global__ void k_rule_labels(const double* err, int np, int nr, DevMesh m, double tau,
                              const int* idx, int* labels) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  int lab = MFB_QNET_CLASSES - 1;
  const double e0 = err[(long long)q * nr];
  if (e0 != e0) {
    lab = -1;  // no reference: no label
  } else {
    for (int r = 0; r < nr; r++)
      if (err[(long long)q * nr + r] <= tau) {
        lab = m.ps_gln[r] - 2;
        break;
      }
  }
  labels[idx[q]] = lab;
}

__global__ void k_fill_int(int* a, int n, int v) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) a[q] = v;
}

#pragma clang fp contract(off)

// Mantic free term (bem_staela3d.f90:228-405) gathered as in
// src/build_lse_mechanics_bem_staela.f90:210-549; I/2 for nodes interior to their first element.
__device__ bool mantic(int m_, double (*ln)[3], double (*lt)[3], double tol, double nu,
                       double* C) {
  // ln, lt indexed 0..m_+1 (0 and m_+1 are the wrap-around copies)
  double lti[kMaxIncid][3], theta[kMaxIncid];
  int tc[kMaxIncid];
  for (int ki = 1; ki <= m_ - 1; ki++) {
    double e1[3] = {lt[ki][0], lt[ki][1], lt[ki][2]}, e3[3] = {ln[ki][0], ln[ki][1], ln[ki][2]}, e2[3];
    e2[0] = e3[1] * e1[2] - e3[2] * e1[1];
    e2[1] = e3[2] * e1[0] - e3[0] * e1[2];
    e2[2] = e3[0] * e1[1] - e3[1] * e1[0];
    for (int kj = 1; kj <= m_; kj++) {
      lti[kj - 1][0] = e1[0] * lt[kj][0] + e1[1] * lt[kj][1] + e1[2] * lt[kj][2];
      lti[kj - 1][1] = e2[0] * lt[kj][0] + e2[1] * lt[kj][1] + e2[2] * lt[kj][2];
      lti[kj - 1][2] = e3[0] * lt[kj][0] + e3[1] * lt[kj][1] + e3[2] * lt[kj][2];
    }
    int nt = 0;
    for (int kj = ki + 1; kj <= m_; kj++)
      if (fabs(lti[kj - 1][2]) <= tol) tc[nt++] = kj;
    if (nt == 0) return false;
    for (int j = 0; j < nt; j++) {
      double a = atan2(lti[tc[j] - 1][1], lti[tc[j] - 1][0]);
      if (a < 0.0) a += 2.0 * kPi;
      theta[tc[j] - 1] = a;
    }
    double mint = theta[tc[0] - 1];
    int mk = tc[0];
    for (int j = 1; j < nt; j++)
      if (theta[tc[j] - 1] < mint) { mint = theta[tc[j] - 1]; mk = tc[j]; }
    for (int c = 0; c < 3; c++) {
      double t = lt[ki + 1][c]; lt[ki + 1][c] = lt[mk][c]; lt[mk][c] = t;
      t = ln[ki + 1][c]; ln[ki + 1][c] = ln[mk][c]; ln[mk][c] = t;
    }
  }
  for (int c = 0; c < 3; c++) {
    ln[0][c] = ln[m_][c]; lt[0][c] = lt[m_][c];
    ln[m_ + 1][c] = ln[1][c]; lt[m_ + 1][c] = lt[1][c];
  }
  double sum_a = 0;
  for (int ki = 1; ki <= m_; ki++) {
    double nx[3];
    nx[0] = ln[ki - 1][1] * ln[ki][2] - ln[ki - 1][2] * ln[ki][1];
    nx[1] = ln[ki - 1][2] * ln[ki][0] - ln[ki - 1][0] * ln[ki][2];
    nx[2] = ln[ki - 1][0] * ln[ki][1] - ln[ki - 1][1] * ln[ki][0];
    double s = nx[0] * lt[ki][0] + nx[1] * lt[ki][1] + nx[2] * lt[ki][2];
    if (s < 0.0) s = -1.0;
    if (s > 0.0) s = 1.0;
    double ndn = ln[ki - 1][0] * ln[ki][0] + ln[ki - 1][1] * ln[ki][1] + ln[ki - 1][2] * ln[ki][2];
    if (ndn > 1.0) ndn = 1.0;
    sum_a = sum_a + s * acos(ndn);
  }
  double cp = 1.0 / (4.0 * kPi) * (2.0 * kPi + sum_a);
  double sb[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int ki = 1; ki <= m_; ki++) {
    double rr[3], rx[3];
    for (int c = 0; c < 3; c++) rr[c] = lt[ki + 1][c] - lt[ki][c];
    rx[0] = rr[1] * ln[ki][2] - rr[2] * ln[ki][1];
    rx[1] = rr[2] * ln[ki][0] - rr[0] * ln[ki][2];
    rx[2] = rr[0] * ln[ki][1] - rr[1] * ln[ki][0];
    for (int c1 = 0; c1 < 3; c1++)
      for (int c2 = 0; c2 < 3; c2++) sb[c1 + 3 * c2] = sb[c1 + 3 * c2] + rx[c1] * ln[ki][c2];
  }
  for (int c1 = 0; c1 < 3; c1++)
    for (int c2 = 0; c2 < 3; c2++) {
      C[c1 + 3 * c2] = -1.0 / (8.0 * kPi * (1.0 - nu)) * sb[c1 + 3 * c2];
      if (c1 == c2) C[c1 + 3 * c2] += cp;
    }
  return true;
}

template <typename T>
__device__ inline void free_term(const DevMesh& m, int i, double nu, T* A, long long lda, T* b,
                                 int* err) {
  if (i >= m.nn) return;
  int q0 = m.inc_ptr[i], q1 = m.inc_ptr[i + 1];
  if (q1 == q0 || m.nmca[i]) return;
  double C[9];
  if (m.inc_k[q0] == 8) {
    for (int c = 0; c < 9; c++) C[c] = (c % 4 == 0) ? 0.5 : 0.0;
  } else {
    int mm = q1 - q0;
    if (mm > kMaxIncid - 2) { atomicExch(err, MFB_ERR_LIMIT); return; }
    double ln[kMaxIncid][3], lt[kMaxIncid][3];
    for (int q = q0; q < q1; q++) {
      double X[27], x[3], T1[3], T2[3], N[3];
      load_X(m, m.inc_e[q], X);
      int k = m.inc_k[q];
      q9_geom(X, kXiQ9[k][0], kXiQ9[k][1], x, T1, T2);
      cross3(T1, T2, N);
      double j = sqrt(dot3(N, N));
      int s = q - q0 + 1;
      for (int c = 0; c < 3; c++) ln[s][c] = N[c] / j;
      // boundary tangent tbp at the node (geometry.f90:657-870)
      const double* Tt = (k == 0 || k == 4 || k == 2 || k == 6) ? T1 : T2;
      double sg = (k == 2 || k == 6 || k == 3 || k == 7) ? -1.0 : 1.0;
      double nt = sqrt(Tt[0] * Tt[0] + Tt[1] * Tt[1] + Tt[2] * Tt[2]);
      for (int c = 0; c < 3; c++) lt[s][c] = sg * (Tt[c] / nt);
    }
    double tol = (m.tol < 1e-12 || m.tol > 1e-3) ? 1e-6 : m.tol;
    if (!mantic(mm, ln, lt, tol, nu, C)) { atomicExch(err, MFB_ERR_GEOMETRY); return; }
  }
  for (int il = 0; il < 3; il++) {
    long long row = 3LL * i + il;
    for (int ik = 0; ik < 3; ik++) {
      long long col = 3LL * i + ik;
      double cv = C[il + 3 * ik];
      if (m.ctype[3 * i + ik] == 0) atomic_add(&b[row], from_real<T>(-(cv * m.cval[3 * i + ik])));
      else atomic_add(&A[row + lda * col], from_real<T>(cv));
    }
  }
}

// Free term of an MCA point: (1/2) u at the point, u interpolated on its element, i.e. (1/2)
// phi_n(xi_i) I on the element's nodes (src/build_lse_mechanics_bem_staela.f90:444-457), scattered by
// the BE-ordinary rule.
template <typename T>
__device__ inline void free_term_mca(const DevMesh& m, int cp, T* A, long long lda, T* b) {
  if (cp >= m.ncp) return;
  const int e = m.cel[cp];
  if (e < 0) return;
  double ph[9];
  phi_q9(m.cxi[2 * cp], m.cxi[2 * cp + 1], ph);
  const int i = m.crow[cp];
  for (int n = 0; n < 9; n++) {
    const int sn = m.conn[9 * e + n];
    const double h = 0.5 * ph[n];
    for (int il = 0; il < 3; il++) {
      const long long row = 3LL * i + il, col = 3LL * sn + il;
      if (m.ctype[3 * sn + il] == 0) atomic_add(&b[row], from_real<T>(-(h * m.cval[3 * sn + il])));
      else atomic_add(&A[row + lda * col], from_real<T>(h));
    }
  }
}

#pragma clang fp contract(fast)

// ------------------------------------------------------------------------------------------------
// Everything that adds to what the tiles have stored, in one launch: subdivided adaptive pairs (a wave
// each, in turn), singular pairs (a workgroup each), the other adaptive pairs (a wave each), free
// terms (a thread each).  The parts are independent (atomic additions), each is a chain of a few
// dependent loads and reductions and none fills the chip on a small mesh: one after the other they
// took 150 of 480 us of a 1,158-DOF assembly (27 us against 61 on a cube of 24 elements,
// 80 against 125 on a sphere of 96, 660 against 930 on an open surface of 26 x 26).  The longest come
// first.
// ------------------------------------------------------------------------------------------------
template <typename T>
struct NearArgs {
  const int *alist, *slist;     // adaptive, singular pairs
  const AdaptGeom* ageo;
  const SingGeom* sgeo;
  int na, ns;
  int tree_wgs;                 // workgroups that take the subdivided pairs
  int nfree, nfree_mca;         // nodes, collocation points whose free terms are added
  double nu;
  T* A;
  long long lda;
  T* b;
  long long* counters;          // quadrature points and leaves of all these pairs are added
  long long sing_points;        // of the singular pairs
  int* err;
  T *ablocks, *sblocks;         // blocks of the pairs (162 values each) instead of A, b
  VecOut<T> vec;                // displacements of their points instead of A, b
};
constexpr int kNearWaves = 4;
static_assert(kNearWaves == kSingWaves, "one workgroup shape");
template <bool H>
struct NearLds {
  union {
    PairLds<kSingWaves> sing;
    struct {
      PairLds<1> pair[kNearWaves];
      WalkLds walk[kNearWaves];
    };
  };
};
template <bool H>
__global__ void __launch_bounds__(kNearWaves* kWave) __attribute__((amdgpu_waves_per_eu(2)))
    k_near(DevMesh m, const QsiParams* __restrict__ qsp, const KernelParams* __restrict__ kpp,
           NearArgs<typename Val<H>::T> a) {
  typedef typename Val<H>::T T;
  __shared__ NearLds<H> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const ConstKP kp = (ConstKP)kpp;
  int wg = blockIdx.x;
  AdaptSum* sum = adapt_sum((AdaptGeom*)a.ageo, a.na);
  // what the records hold already; the subdivided pairs add their own (an addition per pair to one
  // address took longer than the integration at 24,000 pairs)
  if (wg == gridDim.x - 1 && threadIdx.x == 0) {
    atomicAdd((unsigned long long*)&a.counters[0], a.sing_points + (a.na ? sum->points : 0ull));
    if (a.na) atomicAdd((unsigned long long*)&a.counters[1], (unsigned long long)sum->leaves);
  }
  if (wg < a.tree_wgs) {
    const int n = sum->n_tree;
    for (int t = kNearWaves * wg + wave; t < n; t += kNearWaves * a.tree_wgs) {
      wave_lds_fence();
      adaptive_pair<H, true>(m, qsp, kp, a.alist, a.ageo, sum->tree()[t], lds.pair[wave],
                             &lds.walk[wave], a.A, a.lda, a.b, a.counters, a.ablocks, a.vec);
    }
    return;
  }
  wg -= a.tree_wgs;
  if (wg < a.ns) {
    singular_pair<H>(m, kp, a.slist[wg], a.sgeo + wg, lds.sing, a.A, a.lda, a.b,
                     a.sblocks ? a.sblocks + 162LL * wg : (T*)nullptr, a.vec);
    return;
  }
  wg -= a.ns;
  const int adapt_wgs = (a.na + kNearWaves - 1) / kNearWaves;
  if (wg < adapt_wgs) {
    const int q = kNearWaves * wg + wave;
    if (q < a.na && a.ageo[q].gln)
      adaptive_pair<H, false>(m, qsp, kp, a.alist, a.ageo, q, lds.pair[wave], nullptr, a.A, a.lda,
                              a.b, nullptr, a.ablocks, a.vec);
    return;
  }
  wg -= adapt_wgs;
  const int free_wgs = (a.nfree + 255) / 256, i = threadIdx.x;
  if (wg < free_wgs) free_term<T>(m, 256 * wg + i, a.nu, a.A, a.lda, a.b, a.err);
  else free_term_mca<T>(m, 256 * (wg - free_wgs) + i, a.A, a.lda, a.b);
}

}  // namespace mfb

// ================================================================================================
// host side
// ================================================================================================
namespace mfb {

static thread_local char g_err[1024] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
}

// Constant tables of the current device: Gauss-Legendre rules, polar sub-triangles and their points.
static int upload_tables() {
  static bool done = false;
  static int device = -1;
  int dev = 0;
  MFB_HIP(hipGetDevice(&dev));
  if (done && dev == device) return MFB_OK;
  static GLTables t;
  host_gl_tables(&t.x11[0][0], &t.w11[0][0], &t.x01[0][0], &t.w01[0][0]);
  MFB_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_gl), &t, sizeof t));
  static const double xin[9][2] = {{-1, -1}, {1, -1}, {1, 1}, {-1, 1}, {0, -1},
                                   {1, 0},   {0, 1},  {-1, 0}, {0, 0}};
  PolarSet ps[9];
  int np[9];
  std::memset(ps, 0, sizeof ps);
  for (int k = 0; k < 9; k++) {
    ps[k].n = polar_setup_q(xin[k], ps[k].st, ps[k].th, ps[k].thp);
    np[k] = 0;
    for (int s = 0; s < ps[k].n; s++) {
      ps[k].ngt[s] = 5 + (int)std::round(25.0 * (ps[k].th[2 * s + 1] - ps[k].th[2 * s]) / kPi_2);
      np[k] += 15 * ps[k].ngt[s];
    }
    MFB_ARG(np[k] <= kPolarMax, "polar table overflow");
  }
  MFB_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_polar), ps, sizeof ps));
  MFB_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_polar_np), np, sizeof np));
  hipLaunchKernelGGL(k_polar_table, dim3((kPolarMax + 255) / 256, 9), dim3(256), 0, 0);
  MFB_HIP(hipGetLastError());
  MFB_HIP(hipStreamSynchronize(0));
  done = true;
  device = dev;
  return MFB_OK;
}

}  // namespace mfb

namespace mfb {
// scatter tiles of the precalculated classes (k_regular_tile), launched per element colour
struct TileSet {
  int4* d = nullptr;
  size_t cap = 0;                  // tiles the device buffer holds
  // per colour: first tile, tiles; of these the ones that need g alone, and both (in this order, those
  // that need h alone last)
  std::vector<long long> off, cnt, g_only, both;
};
}  // namespace mfb

struct mfb_mesh_s {
  mfb::DevMesh dm;
  mfb::QsiParams qsp, qsp_li;
  int n_cls;
  std::vector<long long> cls_off;  // start of each class list in `lists`
  std::vector<long long> cls_cnt;
  // element colours: elements of one colour share no node, so the pairs of one colour write
  // disjoint entries of A and need no atomics; inside a class list the elements run in
  // (colour, element) order
  int n_colors = 0;
  std::vector<int> ecol, eorder;   // colour of each element; elements in (colour, index) order
  mfb::TileSet tiles;              // of `lists`
  // learned rule choice (mfb_mesh_set_qnet): network, static pair features, the classes and lists
  // of the last assembly, and the judge's result
  mfb_qnet_s* qnet = nullptr;
  float qconf = 0.99f;
  int judge_samples = 0;
  mfb::QsiParams* d_qsp_judge = nullptr;
  // the judge's action (mfb_mesh_set_judge_action): a precalculated rule whose judged pairs miss
  // the tolerance is replaced by the cheapest longer rule that meets it on them (or the adaptive
  // rule) for this and every later assembly of the mesh; promo[r] is that replacement
  int judge_promote = 0;
  std::vector<int> promo;
  int* d_promo = nullptr;
  long long judge_promoted = 0;     // rules promoted by the last assembly
  double judge_first_max = 0;       // the judge's largest error before those promotions
  bool in_redo = false;
  float* feats = nullptr;          // (ne * nn) x MFB_QNET_INPUTS
  int* qcls = nullptr;             // network class per pair
  unsigned char* lcls = nullptr;   // integration class per pair chosen with the network
  int* llists = nullptr;
  std::vector<long long> lcls_off, lcls_cnt;
  mfb::TileSet ltiles;             // of `llists`
  long long l_regular_points = 0;
  bool learned_last = false;
  long long judge_n = 0;
  double judge_max = 0, judge_mean = 0;
  long long judge_ref_n = 0;       // judge pairs where the reference estimator chose a
  double judge_ref_max = 0;        // precalculated rule, and that rule's largest error
  long long* judge_counters = nullptr;  // scratch of the judge's adaptive kernel
  int* judge_err = nullptr;
  // grow-only device workspaces of the per-assembly steps (lists, learned classes, judge): a
  // repeated assembly allocates and frees nothing
  void* ws[12] = {};
  size_t ws_cap[12] = {};
  double *x = nullptr, *cval = nullptr, *elem = nullptr, *ps = nullptr, *nfn = nullptr;
  int *conn = nullptr, *ctype = nullptr, *inc_ptr = nullptr, *inc_e = nullptr, *inc_k = nullptr;
  unsigned char* cls = nullptr;
  int* lists = nullptr;
  // collocation points (device) and host copies of their rows / elements / coordinates
  double *xc = nullptr, *cxi = nullptr;
  int *crow = nullptr, *cel = nullptr;
  unsigned char *nmca = nullptr, *ekind = nullptr;
  int *enode = nullptr, *cx = nullptr, *xnode = nullptr;
  int2* emask = nullptr;
  // interior point sets: the points along a space-filling curve; the node each lies on, -1 none
  int *order = nullptr, *snap = nullptr;
  std::vector<unsigned char> h_kind;   // kNeedH | kNeedG of each element
  bool prezero = false;            // A is reset before the tiles (enode is then ~node throughout)
  mfb::SingGeom* sgeo = nullptr;   // of the singular and the adaptive pairs, in list order
  mfb::AdaptGeom* ageo = nullptr;
  int n_tree = 0;                  // adaptive pairs of `lists` that are subdivided
  long long sing_points = 0;       // quadrature points of the singular pairs
  std::vector<int> h_crow, h_cel;
  std::vector<double> h_xc;
  int n_mca = 0;
  // the geometry and settings it was created from (interior point sets are built from them)
  std::vector<double> h_x, h_cval;
  std::vector<int> h_conn, h_ctype, h_ps;
  double h_tol = 1e-6;
  int* err = nullptr;
  long long* counters = nullptr;  // points, leaves of the adaptive and singular pairs
  mfb::QsiParams* d_qsp = nullptr;     // estimator tables: too large to travel as kernel arguments
  mfb::QsiParams* d_qsp_li = nullptr;
  mfb::KernelParams* d_kp = nullptr;   // kernel constants, read as scalars through the constant cache
  long long decisions = 0;
  long long regular_points = 0;
  // HIP events around the kernel groups of the last assembly (on the caller's stream)
  hipEvent_t ev[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  double last_ms[4] = {0, 0, 0, 0};  // as mfb_mesh_timings gives them
  bool time_groups = false;          // near pairs and free terms launched group by group
  int last_regular_launches = 0;
};

using namespace mfb;

extern "C" const char* mfb_last_error(void) { return g_err; }

template <typename Tp>
static int dalloc(Tp** p, size_t n) {
  MFB_HIP(hipMalloc((void**)p, sizeof(Tp) * (n ? n : 1)));
  return MFB_OK;
}

static void mesh_release(mfb_mesh_s* m) {
  for (hipEvent_t& e : m->ev)
    if (e) (void)hipEventDestroy(e);
  void* ps[] = {m->x,     m->cval,  m->elem,     m->ps,   m->nfn,      m->conn,
                m->ctype, m->inc_ptr, m->inc_e, m->inc_k, m->cls,  m->lists, m->err,
                m->counters, m->d_qsp, m->d_qsp_li, m->d_kp, m->d_qsp_judge, m->feats,
                m->qcls, m->lcls, m->llists, m->judge_counters, m->judge_err,
                m->xc, m->cxi, m->crow, m->cel, m->cx, m->xnode, m->nmca,
                m->ws[0], m->ws[1], m->ws[2], m->ws[3], m->ws[4], m->ws[5], m->ws[6], m->ws[7],
                m->ws[8], m->ws[9], m->ws[10], m->ws[11], m->order, m->snap, m->ageo,
                m->tiles.d, m->ltiles.d, m->d_promo, m->ekind, m->enode, m->emask, m->sgeo};
  for (void* p : ps)
    if (p) (void)hipFree(p);
}

enum MeshWs { MW_OFF, MW_COUNTS, MW_REF, MW_BLK, MW_POS, MW_SAMPLE, MW_ERR, MW_PC, MW_AGEO, MW_JGEO, MW_EXTRA, MW_FIELD };

template <typename P>
static int mesh_ws(mfb_mesh_s* m, int slot, size_t bytes, P** out) {
  if (m->ws_cap[slot] < bytes) {
    if (m->ws[slot]) (void)hipFree(m->ws[slot]);
    m->ws[slot] = nullptr;
    m->ws_cap[slot] = 0;
    MFB_HIP(hipMalloc(&m->ws[slot], bytes));
    m->ws_cap[slot] = bytes;
  }
  *out = reinterpret_cast<P*>(m->ws[slot]);
  return MFB_OK;
}

// k_near; n_tree: how many of the adaptive pairs are subdivided, -1 unknown on the host
template <bool H>
static void launch_near(const DevMesh& d, const QsiParams* qsp, const KernelParams* kpp,
                        NearArgs<typename Val<H>::T> a, int n_tree, hipStream_t s) {
  const int most = n_tree < 0 ? a.na : std::min(n_tree, a.na);
  a.tree_wgs = std::min((most + kNearWaves - 1) / kNearWaves, 512);
  const long long wgs = (long long)a.tree_wgs + a.ns + (a.na + kNearWaves - 1) / kNearWaves +
                        (a.nfree + 255) / 256 + (a.nfree_mca + 255) / 256;
  if (wgs)
    hipLaunchKernelGGL(k_near<H>, dim3((unsigned)wgs), dim3(kNearWaves * kWave), 0, s, d, qsp, kpp, a);
}

// Records of `count` listed adaptive pairs at the tolerance of qsp into geo (adapt_geom_bytes).
static void launch_adapt_geom(const DevMesh& d, const QsiParams* qsp, const int* list, int count,
                              AdaptGeom* geo, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, s, (int*)adapt_sum(geo, count),
                     (int)(sizeof(AdaptSum) / sizeof(int)), 0);
  hipLaunchKernelGGL(k_adapt_geom, dim3((unsigned)((count + 15) / 16)), dim3(kWave), 0, s, d, qsp,
                     list, count, geo);
}

// Geometry records of the singular and the adaptive pairs of the mesh's lists (null stream).
static int make_pair_geom(mfb_mesh_t m) {
  const DevMesh& d = m->dm;
  const long long ns = m->cls_cnt[d.n_ps + 1], na = m->cls_cnt[d.n_ps];
  if (ns) {
    MFB_HIP(hipMalloc((void**)&m->sgeo, sizeof(SingGeom) * (size_t)ns + sizeof(long long) * kSingCounts));
    unsigned long long* np = (unsigned long long*)(m->sgeo + ns);
    MFB_HIP(hipMemset(np, 0, sizeof(long long) * kSingCounts));
    hipLaunchKernelGGL(k_sing_geom, dim3((unsigned)ns), dim3(kWave), 0, 0, d, m->d_qsp_li,
                       m->lists + m->cls_off[d.n_ps + 1], m->sgeo, np);
  }
  if (na) {
    MFB_HIP(hipMalloc((void**)&m->ageo, adapt_geom_bytes((size_t)na)));
    launch_adapt_geom(d, m->d_qsp, m->lists + m->cls_off[d.n_ps], (int)na, m->ageo, 0);
  }
  MFB_HIP(hipGetLastError());
  if (ns) {
    long long np[kSingCounts];
    MFB_HIP(hipMemcpy(np, m->sgeo + ns, sizeof np, hipMemcpyDeviceToHost));
    for (long long n : np) m->sing_points += n;
  }
  if (na)
    MFB_HIP(hipMemcpy(&m->n_tree, &adapt_sum(m->ageo, na)->n_tree, sizeof(int), hipMemcpyDeviceToHost));
  return MFB_OK;
}

// Class lists of the pairs: class-major; inside a class the elements run in (colour, index) order.
// counts: device (ne x (kMaxPrecalsets + 2)) pairs of each class per element; lists: device
// (ne * nn); outputs the host offsets and counts per class and per (class, colour).
static int build_lists(mfb_mesh_t m, const unsigned char* cls, const int* counts, int* lists,
                       std::vector<long long>& cls_off, std::vector<long long>& cls_cnt,
                       TileSet& ts, long long& regular_points, hipStream_t s) {
  const DevMesh& d = m->dm;
  const int ne = d.ne, S = kMaxPrecalsets + 2, nc = m->n_colors;
  std::vector<int> hc((size_t)ne * S);
  MFB_HIP(hipMemcpyAsync(hc.data(), counts, sizeof(int) * ne * S, hipMemcpyDeviceToHost, s));
  MFB_HIP(hipStreamSynchronize(s));
  cls_off.assign(m->n_cls + 1, 0);
  cls_cnt.assign(m->n_cls, 0);
  for (int e = 0; e < ne; e++)
    for (int c = 0; c < m->n_cls; c++) cls_cnt[c] += hc[(size_t)e * S + c];
  for (int c = 0; c < m->n_cls; c++) cls_off[c + 1] = cls_off[c] + cls_cnt[c];
  // off: list start of each (element, class) run; toff: first scatter tile of each (element,
  // precalculated class) run, tiles ordered by colour, then by rule (longest first), then element
  std::vector<long long> off((size_t)2 * ne * S, 0);
  long long* toff = off.data() + (size_t)ne * S;
  std::vector<long long> run(cls_off.begin(), cls_off.end() - 1);
  for (int c = 0; c < m->n_cls; c++)
    for (int q = 0; q < ne; q++) {
      const int e = m->eorder[q];
      off[(size_t)e * S + c] = run[c];
      run[c] += hc[(size_t)e * S + c];
    }
  std::vector<int> rorder(d.n_ps);
  for (int r = 0; r < d.n_ps; r++) rorder[r] = r;
  std::stable_sort(rorder.begin(), rorder.end(),
                   [&](int a, int b) { return d.ps_gln[a] > d.ps_gln[b]; });
  ts.off.assign(nc, 0);
  ts.cnt.assign(nc, 0);
  long long nt = 0;
  ts.g_only.assign(nc, 0);
  ts.both.assign(nc, 0);
  for (int k = 0; k < nc; k++) {
    ts.off[k] = nt;
    for (int kind : {kNeedG, kNeedG | kNeedH, kNeedH}) {
      const long long n0 = nt;
      for (int r : rorder)
        for (int q = 0; q < ne; q++) {
          const int e = m->eorder[q];
          if (m->ecol[e] != k || m->h_kind[e] != kind) continue;
          toff[(size_t)e * S + r] = nt;
          nt += (hc[(size_t)e * S + r] + kTileP - 1) / kTileP;
        }
      if (kind == kNeedG) ts.g_only[k] = nt - n0;
      else if (kind != kNeedH) ts.both[k] = nt - n0;
    }
    ts.cnt[k] = nt - ts.off[k];
  }
  if ((size_t)nt > ts.cap) {
    if (ts.d) (void)hipFree(ts.d);
    ts.d = nullptr;
    ts.cap = 0;
    MFB_HIP(hipMalloc(&ts.d, sizeof(int4) * (size_t)nt));
    ts.cap = (size_t)nt;
  }
  long long* doff = nullptr;
  int rc0 = mesh_ws(m, MW_OFF, sizeof(long long) * 2 * ne * S, &doff);
  if (rc0) return rc0;
  hipError_t he = hipMemcpyAsync(doff, off.data(), sizeof(long long) * 2 * ne * S,
                                 hipMemcpyHostToDevice, s);
  if (he == hipSuccess) {
    hipLaunchKernelGGL(k_fill_lists, dim3(ne), dim3(256), 0, s, d, cls, doff, lists);
    if (nt) hipLaunchKernelGGL(k_fill_tiles, dim3(ne), dim3(64), 0, s, d, counts, doff,
                               doff + (size_t)ne * S, ts.d);
    he = hipGetLastError();
  }
  if (he == hipSuccess) he = hipStreamSynchronize(s);
  if (he != hipSuccess) {
    set_error("build_lists: %s", hipGetErrorString(he));
    return MFB_ERR_HIP;
  }
  regular_points = 0;
  for (int r = 0; r < d.n_ps; r++) regular_points += cls_cnt[r] * d.ps_gln[r] * d.ps_gln[r];
  return MFB_OK;
}

// collocation points of a mesh (host copies; see DevMesh)
struct CollocSet {
  int ncp = 0;
  std::vector<double> xc, cxi;
  std::vector<int> crow, cel;
  std::vector<unsigned char> nmca;
};

static const double kXiQ9H[9][2] = {{-1, -1}, {1, -1}, {1, 1}, {-1, 1}, {0, -1},
                                    {1, 0},   {0, 1},  {-1, 0}, {0, 0}};
static const int kEdgeQ9H[4][3] = {{0, 1, 4}, {1, 2, 5}, {2, 3, 6}, {3, 0, 7}};

// The reference's default BEM formulation of an ordinary boundary
// (src/assign_default_bem_formulation.f90:74-93): nodal SBIE on every node, except the nodes on
// the boundary of the boundary -- element edges that no other element shares
// (lib/fbem/src/data_structures.f90:1620-1640) -- which take SBIE-MCA: one collocation point in
// every element holding the node, at xi_node (1 - delta) (fbem_move_xi1xi2_from_edge,
// lib/fbem/src/geometry.f90:5631-5658; src/build_data_at_collocation_points.f90:125-147), x_i the
// element's position there.  Points are listed node by node; an MCA node's points follow its
// incidences in element order.
static void default_collocation(int nn, int ne, const double* x, const int* conn,
                                const std::vector<int>& ip, const std::vector<int>& ie,
                                const std::vector<int>& ik, double delta, CollocSet& cs) {
  std::map<std::tuple<int, int, int>, int> edges;
  for (int e = 0; e < ne; e++)
    for (int k = 0; k < 4; k++) {
      const int a = conn[9 * e + kEdgeQ9H[k][0]], b = conn[9 * e + kEdgeQ9H[k][1]];
      edges[std::make_tuple(std::min(a, b), std::max(a, b), conn[9 * e + kEdgeQ9H[k][2]])]++;
    }
  cs.nmca.assign(nn, 0);
  for (int e = 0; e < ne; e++)
    for (int k = 0; k < 4; k++) {
      const int a = conn[9 * e + kEdgeQ9H[k][0]], b = conn[9 * e + kEdgeQ9H[k][1]];
      const int c = conn[9 * e + kEdgeQ9H[k][2]];
      if (edges[std::make_tuple(std::min(a, b), std::max(a, b), c)] == 1)
        cs.nmca[a] = cs.nmca[b] = cs.nmca[c] = 1;
    }
  cs.ncp = 0;
  for (int i = 0; i < nn; i++) {
    if (!cs.nmca[i]) {
      for (int c = 0; c < 3; c++) cs.xc.push_back(x[3 * i + c]);
      cs.cxi.push_back(0.0);
      cs.cxi.push_back(0.0);
      cs.crow.push_back(i);
      cs.cel.push_back(-1);
      cs.ncp++;
      continue;
    }
    for (int q = ip[i]; q < ip[i + 1]; q++) {
      const int e = ie[q], k = ik[q];
      const double xi1 = kXiQ9H[k][0] * (1.0 - delta), xi2 = kXiQ9H[k][1] * (1.0 - delta);
      double X[27], xp[3];
      for (int n = 0; n < 9; n++)
        for (int c = 0; c < 3; c++) X[3 * n + c] = x[3 * conn[9 * e + n] + c];
      q9_x(X, xi1, xi2, xp);
      for (int c = 0; c < 3; c++) cs.xc.push_back(xp[c]);
      cs.cxi.push_back(xi1);
      cs.cxi.push_back(xi2);
      cs.crow.push_back(i);
      cs.cel.push_back(e);
      cs.ncp++;
    }
  }
}

// Colours of the elements (no two of a colour share a node), greedily in index order, and where that
// takes more than the four of a structured surface (closed ones: six) once more by saturation
// degree (Brelaz), which is kept if it needs fewer: every colour is a launch, and on a small mesh a
// launch takes its latency (15 us on a cube of 24 elements, 44 on a sphere of 96 elements, each of two
// launches fewer; the assemblies take 155 and 320 us).  Not beyond 4,096 elements, 49,000 unknowns: two
// launches' latency is a thousandth of an assembly there (20 ms for 2,500 elements), the second search
// takes 0.7 ms on the host at 4,056 elements, 2.1 at 9,600 and 3.1 at 21,600.
constexpr int kMaxColors = 64;
static int color_elements(int ne, const int* conn, const std::vector<int>& ip,
                          const std::vector<int>& ie, std::vector<int>& col) {
  auto pick = [&](const std::vector<int>& c, int e) {
    unsigned long long used = 0;
    for (int k = 0; k < 9; k++)
      for (int q = ip[conn[9LL * e + k]]; q < ip[conn[9LL * e + k] + 1]; q++)
        if (c[ie[q]] >= 0) used |= 1ull << c[ie[q]];
    return ~used ? __builtin_ctzll(~used) : kMaxColors;
  };
  int n = 0;
  col.assign(ne, -1);
  for (int e = 0; e < ne; e++) {
    const int c = pick(col, e);
    n = std::max(n, c + 1);
    if (n > kMaxColors) return n;
    col[e] = c;
  }
  if (n <= 4 || ne > 4096) return n;
  std::vector<int> c2(ne, -1), sat(ne, 0);
  std::vector<unsigned long long> seen(ne, 0ull);
  std::vector<std::vector<int>> heap(kMaxColors + 1);   // elements by saturation, stale ones included
  for (int e = ne - 1; e >= 0; e--) heap[0].push_back(e);
  int n2 = 0, top = 0;
  for (int left = ne; left > 0;) {
    while (top > 0 && heap[top].empty()) top--;
    const int e = heap[top].back();
    heap[top].pop_back();
    if (c2[e] >= 0 || sat[e] != top) continue;
    const int c = pick(c2, e);
    n2 = std::max(n2, c + 1);
    if (n2 >= n) return n;
    c2[e] = c;
    left--;
    for (int k = 0; k < 9; k++)
      for (int q = ip[conn[9LL * e + k]]; q < ip[conn[9LL * e + k] + 1]; q++) {
        const int f = ie[q];
        if (c2[f] >= 0 || (seen[f] >> c & 1)) continue;
        seen[f] |= 1ull << c;
        heap[++sat[f]].push_back(f);
        top = std::max(top, sat[f]);
      }
  }
  col.swap(c2);
  return n2;
}

// explicit: a caller-given collocation set (batches of independent pairs); otherwise the
// reference's default formulation with MCA parameter mca_delta.  classify_all = false leaves
// classification and lists to the caller.
static int mesh_create_impl(int nn, int ne, const double* x, const int* conn, const int* ctype,
                            const double* cval, double qsi_relative_error, int qsi_ns_max,
                            int n_precalsets, const int* precalset_gln, double geometric_tolerance,
                            const CollocSet* explicit_cs, double mca_delta, bool classify_all,
                            mfb_mesh_t* out) {
  MFB_ARG(out && x && conn && ctype && cval && precalset_gln, "null argument");
  MFB_ARG(nn > 0 && ne > 0, "empty mesh");
  MFB_ARG(n_precalsets >= 1 && n_precalsets <= kMaxPrecalsets, "1 <= n_precalsets <= 16");
  MFB_ARG(qsi_relative_error >= 1e-15 && qsi_relative_error <= 1e-3,
          "qsi_relative_error must be between 1e-15 and 1e-3 (read_settings.f90:81)");
  MFB_ARG(qsi_ns_max >= 1 && qsi_ns_max <= kMaxNs,
          "qsi_ns_max must be between 1 and 20 (the reference's default is 16)");
  for (int r = 0; r < n_precalsets; r++) {
    // one precalculated rule's kernel values of a pair stay in the LDS of one workgroup
    MFB_ARG(precalset_gln[r] >= 2 && precalset_gln[r] <= kMaxPrecalGln,
            "precalculated rules must be of order 2..21 (the reference's default is 2..9)");
    if (r) MFB_ARG(precalset_gln[r] > precalset_gln[r - 1], "precalsets must be sorted and unique");
  }
  for (long long q = 0; q < 9LL * ne; q++) MFB_ARG(conn[q] >= 0 && conn[q] < nn, "connectivity out of range");
  for (long long q = 0; q < 3LL * nn; q++)
    MFB_ARG(ctype[q] == 0 || ctype[q] == 1 || ctype[q] == 10, "ctype must be 0, 1 or 10");
  int rc = upload_tables();
  if (rc) return rc;

  // node -> (element, local node) incidences, in element order
  std::vector<int> cnt(nn + 1, 0), ip(nn + 1, 0), ie(9LL * ne), ik(9LL * ne);
  for (long long q = 0; q < 9LL * ne; q++) cnt[conn[q]]++;
  for (int i = 0; i < nn; i++) ip[i + 1] = ip[i] + cnt[i];
  std::vector<int> cur(ip.begin(), ip.end() - 1);
  for (int e = 0; e < ne; e++)
    for (int k = 0; k < 9; k++) {
      int j = conn[9 * e + k];
      ie[cur[j]] = e;
      ik[cur[j]] = k;
      cur[j]++;
    }
  CollocSet dcs;
  if (!explicit_cs) default_collocation(nn, ne, x, conn, ip, ie, ik, mca_delta, dcs);
  const CollocSet& cs = explicit_cs ? *explicit_cs : dcs;
  const int ncp = cs.ncp;
  MFB_ARG(ncp > 0 && (long long)ncp * ne < (1LL << 31),
          "collocation points x elements must fit in 31 bits");

  mfb_mesh_s* m = new mfb_mesh_s();
  DevMesh& d = m->dm;
  d.nn = nn;
  d.ne = ne;
  d.ncp = ncp;
  d.n_ps = n_precalsets;
  d.ns_max = qsi_ns_max;
  d.qsi_re = qsi_relative_error;
  d.tol = geometric_tolerance;
  d.ps_off[0] = 0;
  for (int r = 0; r < n_precalsets; r++) {
    d.ps_gln[r] = precalset_gln[r];
    d.ps_off[r + 1] = d.ps_off[r] + precalset_gln[r] * precalset_gln[r];
  }
  d.npts = d.ps_off[n_precalsets];
  host_qsi_params(qsi_relative_error, &m->qsp);
  host_qsi_params(1e-15, &m->qsp_li);
  m->n_cls = n_precalsets + 2;
  m->h_crow = cs.crow;
  m->h_cel = cs.cel;
  m->h_xc = cs.xc;
  m->h_x.assign(x, x + 3LL * nn);
  m->h_cval.assign(cval, cval + 3LL * nn);
  m->h_conn.assign(conn, conn + 9LL * ne);
  m->h_ctype.assign(ctype, ctype + 3LL * nn);
  m->h_ps.assign(precalset_gln, precalset_gln + n_precalsets);
  m->h_tol = geometric_tolerance;
  m->n_mca = 0;
  for (unsigned char f : cs.nmca) m->n_mca += f;

  std::vector<int> ecol;
  const int n_colors = color_elements(ne, conn, ip, ie, ecol);
  const bool color_overflow = n_colors > kMaxColors;
  m->n_colors = n_colors;
  std::vector<int> eorder(ne);
  for (int e = 0; e < ne; e++) eorder[e] = e;
  std::stable_sort(eorder.begin(), eorder.end(), [&](int a, int b) { return ecol[a] < ecol[b]; });

  auto fail = [&](int code) {
    mesh_release(m);
    delete m;
    return code;
  };
  if (color_overflow) {
    set_error("mfb_mesh_create: more than 64 elements share nodes around one element");
    return fail(MFB_ERR_GEOMETRY);
  }
#define TRY(call)               \
  do {                          \
    int rc_ = (call);           \
    if (rc_) return fail(rc_);  \
  } while (0)
#define TRYH(call)                                                                 \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess) {                                                        \
      set_error("%s failed: %s", #call, hipGetErrorString(e_));                    \
      return fail(MFB_ERR_HIP);                                                    \
    }                                                                              \
  } while (0)
  TRY(dalloc(&m->x, 3LL * nn));
  TRY(dalloc(&m->cval, 3LL * nn));
  TRY(dalloc(&m->ctype, 3LL * nn));
  TRY(dalloc(&m->conn, 9LL * ne));
  TRY(dalloc(&m->elem, 8LL * ne));
  TRY(dalloc(&m->ps, (size_t)ne * d.npts * kPsStride));
  TRY(dalloc(&m->nfn, 3LL * nn));
  TRY(dalloc(&m->inc_ptr, nn + 1));
  TRY(dalloc(&m->inc_e, 9LL * ne));
  TRY(dalloc(&m->inc_k, 9LL * ne));
  TRY(dalloc(&m->xc, 3LL * ncp));
  TRY(dalloc(&m->cxi, 2LL * ncp));
  TRY(dalloc(&m->crow, ncp));
  TRY(dalloc(&m->cel, ncp));
  TRY(dalloc(&m->cx, ncp));
  TRY(dalloc(&m->nmca, nn));
  TRY(dalloc(&m->ekind, ne));
  TRY(dalloc(&m->err, 1));
  TRY(dalloc(&m->counters, 2));
  TRY(dalloc(&m->d_qsp, 1));
  TRY(dalloc(&m->d_qsp_li, 1));
  TRY(dalloc(&m->d_kp, 1));
  TRYH(hipMemcpy(m->d_qsp, &m->qsp, sizeof(QsiParams), hipMemcpyHostToDevice));
  for (hipEvent_t& e : m->ev) TRYH(hipEventCreate(&e));
  TRYH(hipMemcpy(m->d_qsp_li, &m->qsp_li, sizeof(QsiParams), hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->x, x, sizeof(double) * 3 * nn, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->cval, cval, sizeof(double) * 3 * nn, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->ctype, ctype, sizeof(int) * 3 * nn, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->conn, conn, sizeof(int) * 9 * ne, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->inc_ptr, ip.data(), sizeof(int) * (nn + 1), hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->inc_e, ie.data(), sizeof(int) * 9 * ne, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->inc_k, ik.data(), sizeof(int) * 9 * ne, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->xc, cs.xc.data(), sizeof(double) * 3 * ncp, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->cxi, cs.cxi.data(), sizeof(double) * 2 * ncp, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->crow, cs.crow.data(), sizeof(int) * ncp, hipMemcpyHostToDevice));
  TRYH(hipMemcpy(m->cel, cs.cel.data(), sizeof(int) * ncp, hipMemcpyHostToDevice));
  {
    std::vector<int> cx(ncp, -1), xnode;
    for (int c = 1; c < ncp && !explicit_cs; c++)
      if (cs.crow[c] == cs.crow[c - 1]) {
        cx[c] = (int)xnode.size();
        xnode.push_back(cs.crow[c]);
      }
    d.nx = (int)xnode.size();
    TRYH(hipMemcpy(m->cx, cx.data(), sizeof(int) * ncp, hipMemcpyHostToDevice));
    TRY(dalloc(&m->xnode, xnode.size()));
    if (d.nx)
      TRYH(hipMemcpy(m->xnode, xnode.data(), sizeof(int) * xnode.size(), hipMemcpyHostToDevice));
  }
  if (cs.nmca.empty()) TRYH(hipMemset(m->nmca, 0, nn));
  else TRYH(hipMemcpy(m->nmca, cs.nmca.data(), nn, hipMemcpyHostToDevice));
  {
    std::vector<unsigned char> ek(ne, 0);
    std::vector<int2> em(ne, make_int2(0, 0));
    for (int e = 0; e < ne; e++) {
      for (int k = 0; k < 27; k++) {
        const long long c = 3LL * conn[9 * e + k / 3] + k % 3;
        ek[e] |= ctype[c] == 0 ? kNeedG : kNeedH;
        if (cval[c] != 0.0) ek[e] |= ctype[c] == 0 ? kNeedH : kNeedG;
        em[e].x |= (ctype[c] == 0) << k;
        em[e].y |= (cval[c] != 0.0) << k;
      }
    }
    m->h_kind = ek;
    TRY(dalloc(&m->emask, ne));
    TRYH(hipMemcpy(m->emask, em.data(), sizeof(int2) * ne, hipMemcpyHostToDevice));
    // the element that stores a node's columns: the one of the lowest colour.  Without one per node, or
    // with a node twice in an element, A is reset and every element adds.
    std::vector<int> en(9LL * ne), owner(nn, -1);
    for (int e = 0; e < ne; e++)
      for (int k = 0; k < 9; k++) {
        for (int l = 0; l < k; l++)
          if (conn[9 * e + k] == conn[9 * e + l]) ek[e] |= kTwice;
        if (ek[e] & kTwice) m->prezero = true;
        int& o = owner[conn[9 * e + k]];
        if (o < 0 || ecol[e] < ecol[o]) o = e;
      }
    for (int i = 0; i < nn; i++) m->prezero = m->prezero || owner[i] < 0;
    for (long long q = 0; q < 9LL * ne; q++)
      en[q] = m->prezero || owner[conn[q]] != q / 9 ? ~conn[q] : conn[q];
    TRY(dalloc(&m->enode, en.size()));
    TRYH(hipMemcpy(m->enode, en.data(), sizeof(int) * en.size(), hipMemcpyHostToDevice));
    TRYH(hipMemcpy(m->ekind, ek.data(), ne, hipMemcpyHostToDevice));
  }
  TRYH(hipMemset(m->err, 0, sizeof(int)));
  TRYH(hipMemset(m->counters, 0, 2 * sizeof(long long)));
  d.x = m->x; d.conn = m->conn; d.ctype = m->ctype; d.cval = m->cval; d.elem = m->elem;
  d.ps = m->ps; d.nfn = m->nfn; d.inc_ptr = m->inc_ptr; d.inc_e = m->inc_e; d.inc_k = m->inc_k;
  d.xc = m->xc; d.cxi = m->cxi; d.crow = m->crow; d.cel = m->cel; d.cx = m->cx; d.xnode = m->xnode;
  d.nmca = m->nmca; d.ekind = m->ekind; d.enode = m->enode; d.emask = m->emask;

  hipLaunchKernelGGL(k_elem_setup, dim3((ne + 63) / 64), dim3(64), 0, 0, d, m->elem);
  TRYH(hipGetLastError());
  long long tot = (long long)ne * d.npts;
  hipLaunchKernelGGL(k_precalc, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, 0, d, m->ps);
  TRYH(hipGetLastError());
  hipLaunchKernelGGL(k_node_normals, dim3((nn + 127) / 128), dim3(128), 0, 0, d, m->nfn);
  TRYH(hipGetLastError());
  m->ecol = ecol;
  m->eorder = eorder;
  m->tiles.off.assign(m->n_colors, 0);
  m->tiles.cnt.assign(m->n_colors, 0);
  m->cls_off.assign(m->n_cls + 1, 0);
  m->cls_cnt.assign(m->n_cls, 0);
  if (classify_all) {
    int* counts = nullptr;
    const int S = kMaxPrecalsets + 2;
    TRY(dalloc(&m->cls, (size_t)ncp * ne));
    TRY(dalloc(&counts, (size_t)ne * S));
    TRYH(hipMemset(counts, 0, sizeof(int) * ne * S));
    hipLaunchKernelGGL(k_classify, dim3(ne), dim3(256), 0, 0, d, m->d_qsp, m->cls, counts);
    TRYH(hipGetLastError());
    TRY(dalloc(&m->lists, (size_t)ncp * ne));
    {
      const int rc = build_lists(m, m->cls, counts, m->lists, m->cls_off, m->cls_cnt, m->tiles,
                                 m->regular_points, 0);
      (void)hipFree(counts);
      if (rc) return fail(rc);
    }
    TRY(make_pair_geom(m));
    // decision checksum (host) and regular-rule quadrature points
    std::vector<unsigned char> hcls((size_t)ncp * ne);
    TRYH(hipMemcpy(hcls.data(), m->cls, hcls.size(), hipMemcpyDeviceToHost));
    long long s = 0;
    for (size_t q = 0; q < hcls.size(); q++) s += (long long)(hcls[q] + 1) * (long long)(q % 97 + 1);
    m->decisions = s;
  }
#undef TRY
#undef TRYH
  *out = m;
  return MFB_OK;
}

extern "C" int mfb_mesh_create(int nn, int ne, const double* x, const int* conn, const int* ctype,
                               const double* cval, double qsi_relative_error, int qsi_ns_max,
                               int n_precalsets, const int* precalset_gln,
                               double geometric_tolerance, mfb_mesh_t* out) {
  // default_mca_boundary_delta (src/assign_default_bem_formulation.f90:40)
  return mesh_create_impl(nn, ne, x, conn, ctype, cval, qsi_relative_error, qsi_ns_max,
                          n_precalsets, precalset_gln, geometric_tolerance, nullptr, 0.05, true, out);
}

extern "C" int mfb_mesh_node_normals(mfb_mesh_t m, double* nfn) {
  MFB_ARG(m && nfn, "null argument");
  MFB_HIP(hipMemcpy(nfn, m->nfn, sizeof(double) * 3 * m->dm.nn, hipMemcpyDeviceToHost));
  return MFB_OK;
}

extern "C" int mfb_mesh_collocation(mfb_mesh_t m, int* ncp, double* xc, int* crow, int* cel) {
  MFB_ARG(m && ncp, "null argument");
  *ncp = m->dm.ncp;
  if (xc) std::memcpy(xc, m->h_xc.data(), sizeof(double) * 3 * m->dm.ncp);
  if (crow) std::memcpy(crow, m->h_crow.data(), sizeof(int) * m->dm.ncp);
  if (cel) std::memcpy(cel, m->h_cel.data(), sizeof(int) * m->dm.ncp);
  return MFB_OK;
}

extern "C" int mfb_mesh_destroy(mfb_mesh_t m) {
  if (!m) return MFB_OK;
  mesh_release(m);
  delete m;
  return MFB_OK;
}

extern "C" int mfb_mesh_pair_classes(mfb_mesh_t m, unsigned char* classes) {
  MFB_ARG(m && classes, "null argument");
  MFB_ARG(m->cls, "this mesh holds no class array");
  MFB_HIP(hipMemcpy(classes, m->cls, (size_t)m->dm.ncp * m->dm.ne, hipMemcpyDeviceToHost));
  return MFB_OK;
}

extern "C" int mfb_mesh_learned_classes(mfb_mesh_t m, unsigned char* classes) {
  MFB_ARG(m && classes, "null argument");
  MFB_ARG(m->lcls && m->learned_last, "the last assembly of this mesh did not use a network");
  MFB_HIP(hipMemcpy(classes, m->lcls, (size_t)m->dm.ncp * m->dm.ne, hipMemcpyDeviceToHost));
  return MFB_OK;
}

extern "C" int mfb_mesh_stats(mfb_mesh_t m, mfb_assembly_stats* s) {
  MFB_ARG(m && s, "null argument");
  const int np = m->dm.n_ps;
  const bool L = m->learned_last;
  const std::vector<long long>& cnt = L ? m->lcls_cnt : m->cls_cnt;
  long long c[2];
  MFB_HIP(hipMemcpy(c, m->counters, sizeof c, hipMemcpyDeviceToHost));
  const long long rp = L ? m->l_regular_points : m->regular_points;
  s->pairs = (long long)m->dm.ncp * m->dm.ne;
  s->singular = cnt[np + 1];
  s->adaptive = cnt[np];
  s->pre = 0;
  for (int r = 0; r < np; r++) s->pre += cnt[r];
  s->points = rp + c[0];
  s->leaves = c[1];
  s->decisions = m->decisions;
  s->regular_points = rp;
  s->learned = L ? 1 : 0;
  s->judge_pairs = m->judge_n;
  s->judge_max_err = m->judge_max;
  s->judge_mean_err = m->judge_mean;
  s->judge_ref_pairs = m->judge_ref_n;
  s->judge_ref_max_err = m->judge_ref_max;
  s->judge_promoted = m->judge_promoted;
  s->judge_first_max_err = m->judge_promoted ? m->judge_first_max : m->judge_max;
  return MFB_OK;
}

template <bool H>
static int run_judge(mfb_mesh_t m, const KernelParams& kp, hipStream_t s);

// k_regular of a rule above 64 KB of LDS (orders >= 14 harmonic, >= 18 static): raise the
// workgroup's dynamic LDS limit (up to the 160 KB of a gfx950 CU)
template <bool H>
static hipError_t set_kreg_lds(size_t lds) {
  hipError_t e = hipFuncSetAttribute((const void*)k_regular<H>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  return e;
}

// Network classes of every pair for this call (k h from the wavenumber kw), then the lists.
static int learned_lists(mfb_mesh_t m, double kw, hipStream_t s) {
  const DevMesh& d = m->dm;
  const long long np = (long long)d.ne * d.ncp;
  hipLaunchKernelGGL(k_set_kh, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, s, d, m->feats, kw);
  int rc = mfb_qnet_classes_device(m->qnet, m->feats, (int)np, m->qconf, m->qcls, s);
  if (rc) return rc;
  int* counts = nullptr;
  rc = mesh_ws(m, MW_COUNTS, sizeof(int) * (size_t)d.ne * (kMaxPrecalsets + 2), &counts);
  if (rc) return rc;
  hipLaunchKernelGGL(k_learned_map, dim3(d.ne), dim3(256), 0, s, d, m->cls, m->qcls, m->d_promo,
                     m->lcls, counts);
  hipError_t he = hipGetLastError();
  if (he != hipSuccess) {
    set_error("k_learned_map: %s", hipGetErrorString(he));
    return MFB_ERR_HIP;
  }
  rc = build_lists(m, m->lcls, counts, m->llists, m->lcls_off, m->lcls_cnt, m->ltiles,
                   m->l_regular_points, s);
  const long long na = rc ? 0 : m->lcls_cnt[d.n_ps];
  if (na) {
    AdaptGeom* geo = nullptr;
    rc = mesh_ws(m, MW_AGEO, adapt_geom_bytes((size_t)na), &geo);
    if (rc) return rc;
    launch_adapt_geom(d, m->d_qsp, m->llists + m->lcls_off[d.n_ps], (int)na, geo, s);
    MFB_HIP(hipGetLastError());
  }
  return rc;
}

// bytes of the extra points' rows
static size_t extra_bytes(mfb_mesh_t m, bool harmonic) {
  return (harmonic ? sizeof(zd) : sizeof(double)) * 9 * (size_t)m->dm.nx * m->dm.nn;
}

// The kernels of one whole-boundary assembly into A, b (scatter mode) on stream s, reading the
// kernel constants at kpp (device): zeroing, the precalculated-rule tiles (one launch per element
// colour), adaptive and singular pairs, free terms.  No host synchronisation and no memset: the
// sequence can be captured into a graph.  extra: workspace of extra_bytes.  events: record the mesh's
// timing events around the kernel groups (not while capturing).
template <bool H>
static int enqueue_scatter(mfb_mesh_t m, const KernelParams* kpp, bool learned, double nu,
                           typename Val<H>::T* A, long long lda, typename Val<H>::T* b,
                           void* extra, hipStream_t s, bool events) {
  typedef typename Val<H>::T T;
  const DevMesh& d = m->dm;
  const int n = 3 * d.nn;
  int* lists = learned ? m->llists : m->lists;
  const std::vector<long long>& cls_off = learned ? m->lcls_off : m->cls_off;
  const std::vector<long long>& cls_cnt = learned ? m->lcls_cnt : m->cls_cnt;
  const TileSet& ts = learned ? m->ltiles : m->tiles;
  if (events) MFB_HIP(hipEventRecord(m->ev[0], s));
  const TileOut<T> out{A, lda, b, (T*)extra};
  if (m->prezero) {
    const long long tot = (long long)n * n, nx = 3LL * d.nx * n;
    // the runtime's fill (6.1 TB/s at 30k) on a stream that is not being captured, a kernel under
    // capture (memset nodes are kept out of graphs) and between padded columns
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    MFB_HIP(hipStreamIsCapturing(s, &cap));
    if (cap == hipStreamCaptureStatusNone && lda == n) {
      MFB_HIP(hipMemsetAsync(A, 0, sizeof(T) * (size_t)tot, s));
    } else {
      const long long nblk = std::min<long long>((tot + 255) / 256, 1 << 14);   // 5.6 TB/s; 1 << 16: 5.1
      hipLaunchKernelGGL(k_zero<T>, dim3((unsigned)nblk), dim3(256), 0, s, A, lda, n);
    }
    if (nx) hipLaunchKernelGGL(k_fill_zero<T>, dim3((unsigned)((nx + 255) / 256)), dim3(256), 0, s, out.X, nx);
  }
  {
    // adaptive and singular pairs are consecutive in the lists
    const int np = m->prezero ? 0 : (int)(cls_cnt[d.n_ps] + cls_cnt[d.n_ps + 1]);
    hipLaunchKernelGGL(k_begin<T>, dim3((unsigned)((np + 3) / 4 + (n + 255) / 256)), dim3(256), 0, s,
                       d, lists + cls_off[d.n_ps], np, out, events ? m->counters : nullptr, m->err);
  }
  if (events) MFB_HIP(hipEventRecord(m->ev[1], s));
  // precalculated rules: one launch per element colour over its tiles (elements of one colour
  // share no node: the pairs of a launch write disjoint entries of A, a plain read-modify-write;
  // the right-hand side keeps atomics)
  if (events) m->last_regular_launches = 0;
  for (int k = 0; k < m->n_colors; k++) {
    if (!ts.cnt[k]) continue;
    if (events) m->last_regular_launches++;
    const int ng = (int)(ts.g_only[k] + ts.both[k]), nh = (int)(ts.cnt[k] - ts.g_only[k]);
    const int run = ng + nh < kRunTiles ? 1 : 32;
    hipLaunchKernelGGL((k_regular_tile<H>), dim3((unsigned)((ng + nh + 8 * run - 1) / (8 * run) * 8 * run)),
                       dim3(kWave), 0, s, d, kpp, lists, ts.d + ts.off[k], (int)ts.g_only[k], nh, ng,
                       run, out);
  }
  if (d.nx)
    hipLaunchKernelGGL(k_fold_extra<T>, dim3((3 * d.nx + 255) / 256, std::min(n, 4096)), dim3(256), 0,
                       s, d, out);
  if (events) MFB_HIP(hipEventRecord(m->ev[2], s));
  NearArgs<T> a{};
  a.alist = lists + cls_off[d.n_ps];
  a.slist = lists + cls_off[d.n_ps + 1];
  a.ageo = learned ? (AdaptGeom*)m->ws[MW_AGEO] : m->ageo;
  a.sgeo = m->sgeo;
  a.na = (int)cls_cnt[d.n_ps];
  a.ns = (int)cls_cnt[d.n_ps + 1];
  a.nfree = d.nn;
  a.nfree_mca = m->n_mca ? d.ncp : 0;
  a.nu = nu;
  a.A = A;
  a.lda = lda;
  a.b = b;
  a.counters = m->counters;
  a.sing_points = m->sing_points;
  a.err = m->err;
  const int n_tree = learned ? -1 : m->n_tree;
  if (!events || !m->time_groups) {
    launch_near<H>(d, m->d_qsp, kpp, a, n_tree, s);
    if (events) MFB_HIP(hipEventRecord(m->ev[3], s));
  } else {   // the same workgroups, group by group
    for (int k = 0; k < 3; k++) {
      NearArgs<T> g = a;
      if (k != 0) g.na = 0;
      if (k != 1) g.ns = 0, g.sing_points = 0;
      if (k != 2) g.nfree = g.nfree_mca = 0;
      launch_near<H>(d, m->d_qsp, kpp, g, n_tree, s);
      MFB_HIP(hipEventRecord(m->ev[3 + k], s));
    }
  }
  MFB_HIP(hipGetLastError());
  return MFB_OK;
}

// blocks == nullptr, vec.out == nullptr: assemble A, b.  blocks: write the 9x3x3 h and g blocks
// of every listed pair to blocks[162*q ...], q = position in the class lists (see
// mfb_pair_blocks).  vec.out: the interior displacements of the collocation points (vec.out is
// overwritten).  Both skip the zeroing of A, the scatter and the free terms.  kw: shear
// wavenumber (0 static), a network feature.
template <bool H>
static int assemble(mfb_mesh_t m, const KernelParams& kp, double nu, double* Araw, long long lda,
                    double* braw, void* stream, double* blocks_raw = nullptr, double kw = 0.0,
                    VecOut<typename Val<H>::T> vec = VecOut<typename Val<H>::T>{}) {
  typedef typename Val<H>::T T;
  T* blocks = (T*)blocks_raw;
  const bool vmode = vec.out != nullptr;
  MFB_ARG(m && ((Araw && braw) || blocks || vmode), "null argument");
  const DevMesh& d = m->dm;
  const int n = 3 * d.nn;
  MFB_ARG(blocks || vmode || lda >= n, "lda < n_dof");
  hipStream_t s = (hipStream_t)stream;
  T* A = (T*)Araw;
  T* b = (T*)braw;
  // kernel constants of this call (ordered before the launches on the same stream)
  MFB_HIP(hipMemcpyAsync(m->d_kp, &kp, sizeof(KernelParams), hipMemcpyHostToDevice, s));
  MFB_HIP(hipStreamSynchronize(s));
  // rule choice: the reference's estimator (classes fixed at mesh creation) or the network
  const bool learned = m->qnet && !blocks && !vmode;
  m->learned_last = learned;
  if (learned) {
    int rc = learned_lists(m, kw, s);
    if (rc) return rc;
  }
  int* lists = learned ? m->llists : m->lists;
  const std::vector<long long>& cls_off = learned ? m->lcls_off : m->cls_off;
  const std::vector<long long>& cls_cnt = learned ? m->lcls_cnt : m->cls_cnt;
  // counters and error flag are cleared by a kernel (no memset nodes if the caller captures)
  if (!blocks && !vmode) {
    void* extra = nullptr;
    int rc = d.nx ? mesh_ws(m, MW_EXTRA, extra_bytes(m, H), &extra) : MFB_OK;
    if (rc == MFB_OK) rc = enqueue_scatter<H>(m, m->d_kp, learned, nu, A, lda, b, extra, s, true);
    if (rc) return rc;
  } else {
    MFB_HIP(hipEventRecord(m->ev[0], s));
    hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, s, m->counters, m->err);
    if (vmode)
      hipLaunchKernelGGL(k_fill_zero<T>, dim3((3 * d.ncp + 255) / 256), dim3(256), 0, s, vec.out,
                         3LL * d.ncp);
    MFB_HIP(hipEventRecord(m->ev[1], s));
    m->last_regular_launches = 0;
    if (vmode) {
      T* field = nullptr;
      const long long nq = (long long)d.ne * d.npts;
      const int rc = mesh_ws(m, MW_FIELD, sizeof(T) * 6 * (size_t)nq, &field);
      if (rc) return rc;
      hipLaunchKernelGGL(k_field<T>, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, s, d, m->d_kp,
                         vec, field);
      // about 8,192 waves; fewer elements per wave would add more sums to the same points
      const long long wv = (d.ncp + 15) / 16;
      const int chunk = (int)std::max<long long>(1, std::max<long long>(wv * d.ne / 8192, (d.ne + 65534) / 65535));
      hipLaunchKernelGGL(k_points<H>, dim3((unsigned)wv, (unsigned)((d.ne + chunk - 1) / chunk)),
                         dim3(kWave), 0, s, d, m->d_kp, m->cls, m->order, field, chunk, vec.out);
      m->last_regular_launches = 1;
    }
    // per-pair blocks: one launch per rule
    for (int r = 0; r < d.n_ps && !vmode; r++) {
      const long long cnt = cls_cnt[r], o = cls_off[r];
      if (!cnt) continue;
      m->last_regular_launches++;
      int P = d.ps_gln[r] * d.ps_gln[r], B = P >= kWave ? 1 : kWave / P;
      long long grid = (cnt + B - 1) / B;
      const size_t lds = kreg_lds_bytes<H>(B * P);
      if (lds > 64 * 1024) MFB_HIP(set_kreg_lds<H>(lds));
      hipLaunchKernelGGL(k_regular<H>, dim3((unsigned)grid), dim3(kWave), lds, s, d, m->d_kp,
                         lists + o, (int)cnt, r, blocks, o);
    }
    MFB_HIP(hipEventRecord(m->ev[2], s));
    NearArgs<T> a{};
    a.alist = lists + cls_off[d.n_ps];
    a.slist = lists + cls_off[d.n_ps + 1];
    a.ageo = m->ageo;
    a.sgeo = m->sgeo;
    a.na = (int)cls_cnt[d.n_ps];
    a.ns = (int)cls_cnt[d.n_ps + 1];
    a.counters = m->counters;
    a.sing_points = m->sing_points;
    a.ablocks = blocks ? blocks + 162 * cls_off[d.n_ps] : nullptr;
    a.sblocks = blocks ? blocks + 162 * cls_off[d.n_ps + 1] : nullptr;
    a.vec = vec;
    launch_near<H>(d, m->d_qsp, m->d_kp, a, m->n_tree, s);
    MFB_HIP(hipEventRecord(m->ev[3], s));
  }
  MFB_HIP(hipGetLastError());
  int herr = 0;
  MFB_HIP(hipMemcpyAsync(&herr, m->err, sizeof(int), hipMemcpyDeviceToHost, s));
  MFB_HIP(hipStreamSynchronize(s));
  {
    float t[5] = {};
    const int groups = m->time_groups && !blocks && !vmode ? 5 : 3;
    for (int q = 0; q < groups; q++) MFB_HIP(hipEventElapsedTime(&t[q], m->ev[q], m->ev[q + 1]));
    m->last_ms[0] = t[1];
    m->last_ms[1] = t[2];
    m->last_ms[2] = t[3];
    m->last_ms[3] = t[0] + t[4];
  }
  if (herr == MFB_ERR_LIMIT) {
    set_error("a free-term node has more incident elements than %d", kMaxIncid - 2);
    return MFB_ERR_LIMIT;
  }
  if (herr == MFB_ERR_GEOMETRY) {
    set_error("the normals/tangents configuration of a free-term node is not valid");
    return MFB_ERR_GEOMETRY;
  }
  if (learned && m->judge_samples > 0) {
    if (!m->in_redo) m->judge_promoted = 0;
    const int rc = run_judge<H>(m, kp, s);
    if (rc || !m->judge_promoted || m->in_redo) return rc;
    // rules were promoted: assemble once more with them (the judge then reports the new choice)
    const double first = m->judge_max;
    m->in_redo = true;
    const int rc2 = assemble<H>(m, kp, nu, Araw, lda, braw, stream, nullptr, kw);
    m->in_redo = false;
    m->judge_first_max = first;
    return rc2;
  }
  m->judge_n = 0;
  m->judge_ref_n = 0;
  return MFB_OK;
}

extern "C" int mfb_mesh_timings(mfb_mesh_t m, double* ms, int* regular_launches) {
  MFB_ARG(m && ms, "null argument");
  for (int q = 0; q < 4; q++) ms[q] = m->last_ms[q];
  if (regular_launches) *regular_launches = m->last_regular_launches;
  return MFB_OK;
}

extern "C" int mfb_mesh_time_groups(mfb_mesh_t m, int on) {
  MFB_ARG(m, "null argument");
  m->time_groups = on != 0;
  return MFB_OK;
}

static KernelParams static_params(double mu, double nu) {
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.harmonic = 0;
  kp.cteu1 = 1.0 / (16.0 * kPi * mu * (1.0 - nu));
  kp.cteu2 = 3.0 - 4.0 * nu;
  kp.ctet1 = -1.0 / (8.0 * kPi * (1.0 - nu));
  kp.ctet2 = 1.0 - 2.0 * nu;
  return kp;
}

extern "C" int mfb_assemble_staela(mfb_mesh_t m, double mu, double nu, double* A, long long lda,
                                   double* b, void* stream) {
  MFB_ARG(mu > 0 && nu < 0.5 && nu > -1.0, "invalid elastic constants");
  return assemble<false>(m, static_params(mu, nu), nu, A, lda, b, stream);
}

extern "C" int mfb_assemble_harela(mfb_mesh_t m, double omega, double lambda_re, double lambda_im,
                                   double mu_re, double mu_im, double rho, double nu, double* A,
                                   long long lda, double* b, void* stream) {
  MFB_ARG(omega > 0 && rho > 0 && mu_re > 0, "invalid harmonic parameters (omega > 0 required)");
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.harmonic = 1;
  host_har_params(lambda_re, lambda_im, mu_re, mu_im, rho, omega, &kp.h);
  return assemble<true>(m, kp, nu, A, lda, b, stream, nullptr, omega * std::sqrt(rho / mu_re));
}

// ------------------------------------------------------------------------------------------------
// Batches of assemblies: many (mesh, material, frequency) jobs enqueued back to back with no host
// synchronisation, and the same sequence captured once into a HIP graph and replayed (with new
// materials / frequencies written into the graph's parameter buffer between launches).  The rule
// choice is the reference's (classes and tiles fixed at mesh creation), so the launch sequence of a
// job does not depend on its frequency.  Every job reads its own kernel constants from one device
// array uploaded by a single host-to-device copy at the start of the sequence.
// ------------------------------------------------------------------------------------------------
static int job_params(const mfb_assembly_job& j, KernelParams* kp) {
  MFB_ARG(j.mesh && j.A && j.b && j.lda >= 3LL * j.mesh->dm.nn, "invalid assembly job");
  MFB_ARG(!j.mesh->qnet, "batched assembly uses the reference rule choice (mesh has a network)");
  if (j.harmonic) {
    MFB_ARG(j.omega > 0 && j.rho > 0 && j.mu_re > 0, "invalid harmonic job parameters");
    std::memset(kp, 0, sizeof *kp);
    kp->harmonic = 1;
    host_har_params(j.lambda_re, j.lambda_im, j.mu_re, j.mu_im, j.rho, j.omega, &kp->h);
  } else {
    MFB_ARG(j.mu_re > 0 && j.nu < 0.5 && j.nu > -1.0, "invalid static job parameters");
    *kp = static_params(j.mu_re, j.nu);
  }
  return MFB_OK;
}

// the jobs' kernels on s: one parameter upload (host_kp pinned), a counter / error reset per
// distinct mesh, then every job's sequence
// bytes of the extra points' rows of a batch (its jobs run one after the other)
static size_t batch_extra_bytes(int njobs, const mfb_assembly_job* jobs) {
  size_t n = 0;
  for (int q = 0; q < njobs; q++)
    if (jobs[q].mesh) n = std::max(n, extra_bytes(jobs[q].mesh, jobs[q].harmonic != 0));
  return n;
}

static int enqueue_batch(int njobs, const mfb_assembly_job* jobs, const KernelParams* host_kp,
                         KernelParams* dev_kp, void* extra, hipStream_t s) {
  MFB_HIP(hipMemcpyAsync(dev_kp, host_kp, sizeof(KernelParams) * njobs, hipMemcpyHostToDevice, s));
  std::vector<mfb_mesh_t> seen;
  for (int q = 0; q < njobs; q++) {
    mfb_mesh_t m = jobs[q].mesh;
    if (std::find(seen.begin(), seen.end(), m) != seen.end()) continue;
    seen.push_back(m);
    hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, s, m->counters, m->err);
  }
  for (int q = 0; q < njobs; q++) {
    const mfb_assembly_job& j = jobs[q];
    const int rc = j.harmonic
        ? enqueue_scatter<true>(j.mesh, dev_kp + q, false, j.nu, (zd*)j.A, j.lda, (zd*)j.b,
                                extra, s, false)
        : enqueue_scatter<false>(j.mesh, dev_kp + q, false, j.nu, j.A, j.lda, j.b, extra,
                                 s, false);
    if (rc) return rc;
  }
  return MFB_OK;
}

// the error flags the kernels of the meshes' last sequences raised (after a synchronisation)
static int batch_errors(int njobs, const mfb_assembly_job* jobs) {
  for (int q = 0; q < njobs; q++) {
    int herr = 0;
    MFB_HIP(hipMemcpy(&herr, jobs[q].mesh->err, sizeof(int), hipMemcpyDeviceToHost));
    if (herr == MFB_ERR_LIMIT) {
      set_error("job %d: a free-term node has more incident elements than %d", q, kMaxIncid - 2);
      return MFB_ERR_LIMIT;
    }
    if (herr == MFB_ERR_GEOMETRY) {
      set_error("job %d: the normals/tangents configuration of a free-term node is not valid", q);
      return MFB_ERR_GEOMETRY;
    }
  }
  return MFB_OK;
}

struct mfb_batch_graph_s {
  std::vector<mfb_assembly_job> jobs;
  KernelParams* host_kp = nullptr;   // pinned: the graph's copy node reads it at every launch
  KernelParams* dev_kp = nullptr;
  void* extra = nullptr;             // rows of the extra collocation points
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipStream_t cap = nullptr;
};

static void batch_graph_release(mfb_batch_graph_s* g) {
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  if (g->cap) (void)hipStreamDestroy(g->cap);
  if (g->host_kp) (void)hipHostFree(g->host_kp);
  if (g->dev_kp) (void)hipFree(g->dev_kp);
  if (g->extra) (void)hipFree(g->extra);
  delete g;
}

extern "C" int mfb_assemble_batch(int njobs, const mfb_assembly_job* jobs, void* stream) {
  MFB_ARG(njobs > 0 && jobs, "null argument");
  hipStream_t s = (hipStream_t)stream;
  KernelParams *hk = nullptr, *dk = nullptr;
  MFB_HIP(hipHostMalloc((void**)&hk, sizeof(KernelParams) * njobs));
  struct Free {
    KernelParams *h, *d;
    void* x;
    ~Free() { if (h) (void)hipHostFree(h); if (d) (void)hipFree(d); if (x) (void)hipFree(x); }
  } fr{hk, nullptr, nullptr};
  for (int q = 0; q < njobs; q++) {
    const int rc = job_params(jobs[q], hk + q);
    if (rc) return rc;
  }
  MFB_HIP(hipMalloc(&dk, sizeof(KernelParams) * njobs));
  fr.d = dk;
  const size_t xb = batch_extra_bytes(njobs, jobs);
  if (xb) MFB_HIP(hipMalloc(&fr.x, xb));
  int rc = enqueue_batch(njobs, jobs, hk, dk, fr.x, s);
  if (rc) return rc;
  MFB_HIP(hipStreamSynchronize(s));
  return batch_errors(njobs, jobs);
}

extern "C" int mfb_batch_graph_create(int njobs, const mfb_assembly_job* jobs,
                                      mfb_batch_graph_t* out) {
  MFB_ARG(njobs > 0 && jobs && out, "null argument");
  auto* g = new mfb_batch_graph_s();
  auto fail = [&](int rc) { batch_graph_release(g); return rc; };
  g->jobs.assign(jobs, jobs + njobs);
  if (hipHostMalloc((void**)&g->host_kp, sizeof(KernelParams) * njobs) != hipSuccess ||
      hipMalloc(&g->dev_kp, sizeof(KernelParams) * njobs) != hipSuccess ||
      hipStreamCreateWithFlags(&g->cap, hipStreamNonBlocking) != hipSuccess) {
    set_error("mfb_batch_graph_create: allocation failed");
    return fail(MFB_ERR_HIP);
  }
  for (int q = 0; q < njobs; q++) {
    const int rc = job_params(jobs[q], g->host_kp + q);
    if (rc) return fail(rc);
  }
  const size_t xb = batch_extra_bytes(njobs, jobs);
  if (xb && hipMalloc(&g->extra, xb) != hipSuccess) {
    set_error("mfb_batch_graph_create: allocation failed");
    return fail(MFB_ERR_HIP);
  }
  hipError_t he = hipStreamBeginCapture(g->cap, hipStreamCaptureModeThreadLocal);
  if (he != hipSuccess) {
    set_error("hipStreamBeginCapture: %s", hipGetErrorString(he));
    return fail(MFB_ERR_HIP);
  }
  const int rc = enqueue_batch(njobs, jobs, g->host_kp, g->dev_kp, g->extra, g->cap);
  he = hipStreamEndCapture(g->cap, &g->graph);
  if (rc) return fail(rc);
  if (he == hipSuccess) he = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
  if (he != hipSuccess) {
    set_error("graph capture: %s", hipGetErrorString(he));
    return fail(MFB_ERR_HIP);
  }
  *out = g;
  return MFB_OK;
}

extern "C" int mfb_batch_graph_set_params(mfb_batch_graph_t g, int njobs,
                                          const mfb_assembly_job* jobs) {
  MFB_ARG(g && jobs && njobs == (int)g->jobs.size(), "job count differs from the graph's");
  for (int q = 0; q < njobs; q++) {
    const mfb_assembly_job &a = jobs[q], &c = g->jobs[q];
    MFB_ARG(a.mesh == c.mesh && a.A == c.A && a.b == c.b && a.lda == c.lda &&
                a.harmonic == c.harmonic,
            "a job's mesh, buffers or kind differ from the captured graph's");
  }
  // the previous launch may still read the parameters: wait for it before rewriting them
  MFB_HIP(hipStreamSynchronize(g->cap));
  for (int q = 0; q < njobs; q++) {
    KernelParams kp;
    const int rc = job_params(jobs[q], &kp);
    if (rc) return rc;
    g->host_kp[q] = kp;
    g->jobs[q] = jobs[q];
  }
  return MFB_OK;
}

extern "C" int mfb_batch_graph_launch(mfb_batch_graph_t g, void* stream) {
  MFB_ARG(g, "null argument");
  hipStream_t s = stream ? (hipStream_t)stream : g->cap;
  MFB_HIP(hipGraphLaunch(g->exec, s));
  if (s != g->cap) {   // set_params waits on the capture stream: order it after this launch
    hipEvent_t ev;
    MFB_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    MFB_HIP(hipEventRecord(ev, s));
    MFB_HIP(hipStreamWaitEvent(g->cap, ev, 0));
    MFB_HIP(hipEventDestroy(ev));
  }
  return MFB_OK;
}

extern "C" int mfb_batch_graph_check(mfb_batch_graph_t g) {
  MFB_ARG(g, "null argument");
  MFB_HIP(hipStreamSynchronize(g->cap));
  MFB_HIP(hipDeviceSynchronize());
  return batch_errors((int)g->jobs.size(), g->jobs.data());
}

extern "C" int mfb_batch_graph_destroy(mfb_batch_graph_t g) {
  if (!g) return MFB_OK;
  (void)hipStreamSynchronize(g->cap);
  batch_graph_release(g);
  return MFB_OK;
}

// ------------------------------------------------------------------------------------------------
// Learned rule choice: features and labels of listed pairs (pair id = e * nn + i)
// ------------------------------------------------------------------------------------------------
__global__ void k_gather_cls(const unsigned char* cls, const int* pairs, int np, int* out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < np) out[q] = cls[pairs[q]];
}

__global__ void k_scatter_rows(const double* src, int np, int nr, const int* idx, double* dst) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)np * nr) return;
  const int q = (int)(t / nr), r = (int)(t % nr);
  dst[(long long)idx[q] * nr + r] = src[t];
}

__global__ void k_fill_double(double* a, long long n, double v) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) a[q] = v;
}

// err (np x n_ps, device): error of every precalculated rule of the listed (non-singular) pairs
// against the adaptive rule run with the estimator tables d_qsp_ref
template <bool H>
static int rule_errors(mfb_mesh_t m, const KernelParams& kp, const int* dlist, int np,
                       const QsiParams* d_qsp_ref, double* err, long long* counters, int* errflag,
                       hipStream_t s) {
  typedef typename Val<H>::T T;
  const DevMesh& d = m->dm;
  T *ref = nullptr, *blk = nullptr;
  int rc = mesh_ws(m, MW_REF, sizeof(T) * 162 * (size_t)np, &ref);
  if (!rc) rc = mesh_ws(m, MW_BLK, sizeof(T) * 162 * (size_t)np, &blk);
  AdaptGeom* geo = nullptr;
  if (!rc) rc = mesh_ws(m, MW_JGEO, adapt_geom_bytes((size_t)np), &geo);
  if (rc) return rc;
  hipError_t he = hipMemcpyAsync(m->d_kp, &kp, sizeof(KernelParams), hipMemcpyHostToDevice, s);
  if (he == hipSuccess) he = hipStreamSynchronize(s);
  if (he == hipSuccess) {
    hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, s, counters, errflag);
    launch_adapt_geom(d, d_qsp_ref, dlist, np, geo, s);
    NearArgs<T> a{};
    a.alist = dlist;
    a.ageo = geo;
    a.na = np;
    a.counters = counters;
    a.ablocks = ref;
    launch_near<H>(d, d_qsp_ref, m->d_kp, a, -1, s);
    for (int r = 0; r < d.n_ps; r++) {
      const int P = d.ps_gln[r] * d.ps_gln[r], B = P >= kWave ? 1 : kWave / P;
      hipLaunchKernelGGL(k_regular<H>, dim3((unsigned)((np + B - 1) / B)), dim3(kWave),
                         kreg_lds_bytes<H>(B * P), s, d, m->d_kp, dlist, np, r, blk, 0LL);
      hipLaunchKernelGGL(k_block_err<T>, dim3((unsigned)np), dim3(kWave), 0, s, ref, blk, d.n_ps,
                         r, err);
    }
    he = hipGetLastError();
  }
  if (he == hipSuccess) he = hipStreamSynchronize(s);
  if (he != hipSuccess) {
    set_error("rule_errors: %s", hipGetErrorString(he));
    rc = MFB_ERR_HIP;
  }
  return rc;
}

// The judge of the learned rule choice: an evenly spaced sample of the pairs the network gave a
// precalculated rule is integrated with the adaptive rule at the judge's tolerance; the sample's
// largest and mean block errors of the rules actually used are kept for mfb_mesh_stats.
template <bool H>
static int run_judge(mfb_mesh_t m, const KernelParams& kp, hipStream_t s) {
  const DevMesh& d = m->dm;
  const long long total = m->lcls_off[d.n_ps];
  m->judge_n = 0;
  m->judge_max = 0;
  m->judge_mean = 0;
  m->judge_ref_n = 0;
  m->judge_ref_max = 0;
  if (total == 0) return MFB_OK;
  const int K = (int)std::min<long long>(m->judge_samples, total);
  std::vector<long long> pos(K);
  std::vector<int> rk(K);
  for (int k = 0; k < K; k++) {
    pos[k] = std::min(total - 1, (long long)(((double)k + 0.5) * (double)total / (double)K));
    int r = 0;
    while (r + 1 < d.n_ps && pos[k] >= m->lcls_off[r + 1]) r++;
    rk[k] = r;
  }
  long long* dpos = nullptr;
  int* dsample = nullptr;
  double* err = nullptr;
  int rc = mesh_ws(m, MW_POS, sizeof(long long) * K, &dpos);
  if (!rc) rc = mesh_ws(m, MW_SAMPLE, sizeof(int) * K, &dsample);
  if (!rc) rc = mesh_ws(m, MW_ERR, sizeof(double) * (size_t)K * d.n_ps, &err);
  if (rc) return rc;
  hipError_t he = hipMemcpyAsync(dpos, pos.data(), sizeof(long long) * K, hipMemcpyHostToDevice, s);
  if (he == hipSuccess) {
    hipLaunchKernelGGL(k_gather_list, dim3((K + 255) / 256), dim3(256), 0, s, m->llists, dpos, K,
                       dsample);
    rc = rule_errors<H>(m, kp, dsample, K, m->d_qsp_judge, err, m->judge_counters, m->judge_err,
                        s);
  } else {
    set_error("run_judge: %s", hipGetErrorString(he));
    rc = MFB_ERR_HIP;
  }
  // the reference estimator's rule for the same pairs (when it is a precalculated one)
  std::vector<int> pc(K, -1);
  int* dpc = nullptr;
  if (rc == MFB_OK) {
    rc = mesh_ws(m, MW_PC, sizeof(int) * K, &dpc);
    if (rc) return rc;
    {
      hipLaunchKernelGGL(k_gather_cls, dim3((K + 255) / 256), dim3(256), 0, s, m->cls, dsample, K, dpc);
      he = hipMemcpyAsync(pc.data(), dpc, sizeof(int) * K, hipMemcpyDeviceToHost, s);
    }
    if (he == hipSuccess) he = hipStreamSynchronize(s);
    if (he != hipSuccess) {
      set_error("run_judge: %s", hipGetErrorString(he));
      rc = MFB_ERR_HIP;
    }
  }
  if (rc == MFB_OK) {
    std::vector<double> he_(static_cast<size_t>(K) * d.n_ps);
    he = hipMemcpy(he_.data(), err, sizeof(double) * he_.size(), hipMemcpyDeviceToHost);
    if (he != hipSuccess) {
      set_error("run_judge: %s", hipGetErrorString(he));
      rc = MFB_ERR_HIP;
    } else {
      double mx = 0, sum = 0, pmx = 0;
      long long pn = 0, nk = 0;
      for (int k = 0; k < K; k++) {
        const double e = he_[(size_t)k * d.n_ps + rk[k]];
        if (e != e) continue;  // no reference for this pair
        nk++;
        mx = std::max(mx, e);
        sum += e;
        if (pc[k] >= 0 && pc[k] < d.n_ps) {
          pmx = std::max(pmx, he_[(size_t)k * d.n_ps + pc[k]]);
          pn++;
        }
      }
      m->judge_n = nk;
      m->judge_max = mx;
      m->judge_mean = nk ? sum / nk : 0.0;
      m->judge_ref_n = pn;
      m->judge_ref_max = pmx;
      if (m->judge_promote && !m->in_redo) {
        // a rule whose judged pairs miss the tolerance: the cheapest longer rule that meets it on
        // all of them, else the adaptive rule; the promotion applies to the network classes that
        // map to the rule (promo composes with earlier promotions)
        const double tol = d.qsi_re;
        bool changed = false;
        for (int r = 0; r < d.n_ps; r++) {
          double worst = 0;
          bool any = false;
          for (int k = 0; k < K; k++) {
            const double e = he_[(size_t)k * d.n_ps + r];
            if (rk[k] != r || e != e) continue;
            any = true;
            worst = std::max(worst, e);
          }
          if (!any || worst <= tol) continue;
          int to = d.n_ps;   // adaptive
          for (int r2 = 0; r2 < d.n_ps && to == d.n_ps; r2++) {
            if (d.ps_gln[r2] <= d.ps_gln[r]) continue;
            bool ok = true;
            for (int k = 0; k < K && ok; k++) {
              const double e = he_[(size_t)k * d.n_ps + r2];
              if (rk[k] == r && e == e && e > tol) ok = false;
            }
            if (ok) to = r2;
          }
          for (int q = 0; q < d.n_ps; q++)
            if (m->promo[q] == r) m->promo[q] = to;
          m->judge_promoted++;
          changed = true;
        }
        if (changed) {
          he = hipMemcpy(m->d_promo, m->promo.data(), sizeof(int) * d.n_ps, hipMemcpyHostToDevice);
          if (he != hipSuccess) {
            set_error("run_judge: %s", hipGetErrorString(he));
            rc = MFB_ERR_HIP;
          }
        }
      }
    }
  }
  return rc;
}

extern "C" int mfb_mesh_set_qnet(mfb_mesh_t m, mfb_qnet_t q, float confidence,
                                 double judge_qsi_relative_error, int judge_samples) {
  MFB_ARG(m, "null mesh");
  if (!q) {
    m->qnet = nullptr;
    return MFB_OK;
  }
  MFB_ARG(confidence > 0.f && confidence <= 1.f, "confidence must be in (0, 1]");
  MFB_ARG(judge_samples >= 0 && judge_qsi_relative_error > 0 && judge_qsi_relative_error < 1,
          "judge_samples >= 0 and 0 < judge_qsi_relative_error < 1 required");
  const DevMesh& d = m->dm;
  const long long np = (long long)d.ne * d.ncp;
  MFB_ARG(m->cls, "this mesh holds no class array");
  if (!m->feats) {
    MFB_HIP(hipMalloc(&m->feats, sizeof(float) * MFB_QNET_INPUTS * (size_t)np));
    MFB_HIP(hipMalloc(&m->qcls, sizeof(int) * (size_t)np));
    MFB_HIP(hipMalloc(&m->lcls, (size_t)np));
    MFB_HIP(hipMalloc(&m->llists, sizeof(int) * (size_t)np));
    MFB_HIP(hipMalloc(&m->d_qsp_judge, sizeof(QsiParams)));
    MFB_HIP(hipMalloc(&m->judge_counters, 2 * sizeof(long long)));
    MFB_HIP(hipMalloc(&m->judge_err, sizeof(int)));
    MFB_HIP(hipMalloc(&m->d_promo, sizeof(int) * kMaxPrecalsets));
    hipLaunchKernelGGL(k_all_features, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, 0, d,
                       m->feats);
    MFB_HIP(hipGetLastError());
    MFB_HIP(hipDeviceSynchronize());
  }
  QsiParams hq;
  host_qsi_params(judge_qsi_relative_error, &hq);
  MFB_HIP(hipMemcpy(m->d_qsp_judge, &hq, sizeof(QsiParams), hipMemcpyHostToDevice));
  m->qnet = q;
  m->qconf = confidence;
  m->judge_samples = judge_samples;
  // a new network starts without promotions
  m->promo.resize(d.n_ps);
  for (int r = 0; r < d.n_ps; r++) m->promo[r] = r;
  MFB_HIP(hipMemcpy(m->d_promo, m->promo.data(), sizeof(int) * d.n_ps, hipMemcpyHostToDevice));
  return MFB_OK;
}

extern "C" int mfb_mesh_set_judge_action(mfb_mesh_t m, int promote) {
  MFB_ARG(m && m->qnet, "the mesh has no network (mfb_mesh_set_qnet first)");
  MFB_ARG(m->judge_samples > 0 || !promote, "the judge samples no pairs (judge_samples = 0)");
  m->judge_promote = promote ? 1 : 0;
  return MFB_OK;
}

template <bool H>
static int pair_labels(mfb_mesh_t m, const KernelParams& kp, const int* pairs, int np, double tau,
                       int* labels, double* errors, hipStream_t s) {
  MFB_ARG(m && pairs && labels && np > 0 && tau > 0, "bad argument");
  const DevMesh& d = m->dm;
  const int nr = d.n_ps;
  std::vector<int> hp(np), hc(np);
  int* dcls = nullptr;
  MFB_HIP(hipMalloc(&dcls, sizeof(int) * np));
  hipLaunchKernelGGL(k_gather_cls, dim3((np + 255) / 256), dim3(256), 0, s, m->cls, pairs, np, dcls);
  MFB_HIP(hipMemcpyAsync(hc.data(), dcls, sizeof(int) * np, hipMemcpyDeviceToHost, s));
  MFB_HIP(hipMemcpyAsync(hp.data(), pairs, sizeof(int) * np, hipMemcpyDeviceToHost, s));
  MFB_HIP(hipStreamSynchronize(s));
  (void)hipFree(dcls);
  std::vector<int> flist, fidx;
  for (int q = 0; q < np; q++)
    if (hc[q] != d.n_ps + 1) {
      flist.push_back(hp[q]);
      fidx.push_back(q);
    }
  const int nf = (int)flist.size();
  hipLaunchKernelGGL(k_fill_int, dim3((np + 255) / 256), dim3(256), 0, s, labels, np, -1);
  if (errors)
    hipLaunchKernelGGL(k_fill_double, dim3((unsigned)(((long long)np * nr + 255) / 256)), dim3(256),
                       0, s, errors, (long long)np * nr, -1.0);
  if (nf == 0) {
    MFB_HIP(hipStreamSynchronize(s));
    return MFB_OK;
  }
  int *dl = nullptr, *di = nullptr;
  double* err = nullptr;
  MFB_HIP(hipMalloc(&dl, sizeof(int) * nf));
  MFB_HIP(hipMalloc(&di, sizeof(int) * nf));
  MFB_HIP(hipMalloc(&err, sizeof(double) * (size_t)nf * nr));
  MFB_HIP(hipMemcpyAsync(dl, flist.data(), sizeof(int) * nf, hipMemcpyHostToDevice, s));
  MFB_HIP(hipMemcpyAsync(di, fidx.data(), sizeof(int) * nf, hipMemcpyHostToDevice, s));
  int rc = rule_errors<H>(m, kp, dl, nf, m->d_qsp, err, m->counters, m->err, s);
  if (rc == MFB_OK) {
    hipLaunchKernelGGL(k_rule_labels, dim3((nf + 255) / 256), dim3(256), 0, s, err, nf, nr, d, tau,
                       di, labels);
    if (errors)
      hipLaunchKernelGGL(k_scatter_rows, dim3((unsigned)(((long long)nf * nr + 255) / 256)),
                         dim3(256), 0, s, err, nf, nr, di, errors);
    hipError_t he = hipGetLastError();
    if (he == hipSuccess) he = hipStreamSynchronize(s);
    if (he != hipSuccess) {
      set_error("pair_labels: %s", hipGetErrorString(he));
      rc = MFB_ERR_HIP;
    }
  }
  (void)hipFree(dl);
  (void)hipFree(di);
  (void)hipFree(err);
  return rc;
}

extern "C" int mfb_mesh_pair_features(mfb_mesh_t m, const int* pairs, int np, double wavenumber,
                                      float* feats, void* stream) {
  MFB_ARG(m && pairs && feats && np > 0 && wavenumber >= 0, "bad argument");
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_pair_features, dim3((np + 127) / 128), dim3(128), 0, s, m->dm, pairs, np,
                     wavenumber, feats);
  MFB_HIP(hipGetLastError());
  MFB_HIP(hipStreamSynchronize(s));
  return MFB_OK;
}

extern "C" int mfb_mesh_pair_labels_staela(mfb_mesh_t m, double mu, double nu, const int* pairs,
                                           int np, double tau, int* labels, double* errors,
                                           void* stream) {
  MFB_ARG(mu > 0 && nu < 0.5 && nu > -1.0, "invalid elastic constants");
  return pair_labels<false>(m, static_params(mu, nu), pairs, np, tau, labels, errors,
                            (hipStream_t)stream);
}

extern "C" int mfb_mesh_pair_labels_harela(mfb_mesh_t m, double omega, double lambda_re,
                                           double lambda_im, double mu_re, double mu_im,
                                           double rho, const int* pairs, int np, double tau,
                                           int* labels, double* errors, void* stream) {
  MFB_ARG(omega > 0 && rho > 0 && mu_re > 0, "invalid harmonic parameters (omega > 0 required)");
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.harmonic = 1;
  host_har_params(lambda_re, lambda_im, mu_re, mu_im, rho, omega, &kp.h);
  return pair_labels<true>(m, kp, pairs, np, tau, labels, errors, (hipStream_t)stream);
}

// Host scatter of one pair block (src/assemble_bem_staela_equation.f90:69-98).
template <typename V>
static void scatter_host(const int* ctype, const double* cval, const double* nfn, int reversion,
                         int ncol, const int* en, const V* h, const V* g, V* A, long long lda,
                         V* b) {
  for (int il = 0; il < 3; il++) {
    long long row = 3LL * ncol + il;
    for (int ik = 0; ik < 3; ik++)
      for (int kn = 0; kn < 9; kn++) {
        int sn = en[kn];
        long long col = 3LL * sn + ik;
        int o = kn + 9 * il + 27 * ik;
        int ct = ctype[3 * sn + ik];
        double cv = cval[3 * sn + ik];
        switch (ct) {
          case 0:
            A[row + lda * col] -= g[o];
            b[row] -= h[o] * cv;
            break;
          case 1:
            A[row + lda * col] += h[o];
            b[row] += g[o] * cv;
            break;
          default:
            A[row + lda * col] += h[o];
            if (!reversion) b[row] += g[o] * cv * nfn[3 * sn + ik];
            else b[row] -= g[o] * cv * nfn[3 * sn + ik];
        }
      }
  }
}

extern "C" int mfb_assemble_bem_staela_equation(int nn, const int* ctype, const double* cval,
                                                const double* node_normal, int reversion,
                                                int node_col, const int* enodes, const double* h,
                                                const double* g, double* A, long long lda,
                                                double* b) {
  MFB_ARG(ctype && cval && node_normal && enodes && h && g && A && b, "null argument");
  MFB_ARG(node_col >= 0 && node_col < nn && lda >= 3LL * nn, "index out of range");
  for (int k = 0; k < 9; k++) MFB_ARG(enodes[k] >= 0 && enodes[k] < nn, "element node out of range");
  scatter_host<double>(ctype, cval, node_normal, reversion, node_col, enodes, h, g, A, lda, b);
  return MFB_OK;
}

extern "C" int mfb_assemble_bem_harela_equation(int nn, const int* ctype, const double* cval,
                                                const double* node_normal, int reversion,
                                                int node_col, const int* enodes, const double* h,
                                                const double* g, double* A, long long lda,
                                                double* b) {
  MFB_ARG(ctype && cval && node_normal && enodes && h && g && A && b, "null argument");
  MFB_ARG(node_col >= 0 && node_col < nn && lda >= 3LL * nn, "index out of range");
  for (int k = 0; k < 9; k++) MFB_ARG(enodes[k] >= 0 && enodes[k] < nn, "element node out of range");
  typedef std::complex<double> z;
  scatter_host<z>(ctype, cval, node_normal, reversion, node_col, enodes, (const z*)h, (const z*)g,
                  (z*)A, lda, (z*)b);
  return MFB_OK;
}

// The BE-ordinary scatter with the reference's own DOF tables (node%row, node%col, ctype, cvalue,
// n_fn of src/assemble_bem_{staela,harela}_equation.f90:69-113): rows[il] = equation of direction
// il of the collocation node; cols[6 kn + k] = column of unknown k of element node kn (k < 3:
// u_k, k >= 3: t_{k-3}; -1 where the node has none).  ctype 2/3 (local-axes conditions: u and t
// both unknown, harmonic only) put h in the u column and -g in the t column.
template <typename V>
static int scatter_tables(int n_el_nodes, const int* rows, const int* cols, const int* ctype,
                          const V* cval, const double* n_fn, int reversion, const V* h, const V* g,
                          V* A, long long lda, V* b, bool allow_local) {
  const int ne = n_el_nodes;
  for (int il = 0; il < 3; il++) {
    const long long row = rows[il];
    for (int ik = 0; ik < 3; ik++)
      for (int kn = 0; kn < ne; kn++) {
        const int o = kn + ne * il + 3 * ne * ik;
        const int ct = ctype[3 * kn + ik];
        const V cv = cval[3 * kn + ik];
        const long long cu = cols[6 * kn + ik], ct_col = cols[6 * kn + 3 + ik];
        switch (ct) {
          case 0:
            if (ct_col < 0) return MFB_ERR_ARG;
            A[row + lda * ct_col] -= g[o];
            b[row] -= h[o] * cv;
            break;
          case 1:
            if (cu < 0) return MFB_ERR_ARG;
            A[row + lda * cu] += h[o];
            b[row] += g[o] * cv;
            break;
          case 10:
            if (cu < 0) return MFB_ERR_ARG;
            A[row + lda * cu] += h[o];
            if (!reversion) b[row] += g[o] * cv * n_fn[3 * kn + ik];
            else b[row] -= g[o] * cv * n_fn[3 * kn + ik];
            break;
          case 2:
          case 3:
            if (!allow_local || cu < 0 || ct_col < 0) return MFB_ERR_ARG;
            A[row + lda * cu] += h[o];
            A[row + lda * ct_col] -= g[o];
            break;
          default:
            return MFB_ERR_ARG;
        }
      }
  }
  return MFB_OK;
}

extern "C" int mfb_scatter_bem_staela_equation(int n_el_nodes, const int* rows, const int* cols,
                                               const int* ctype, const double* cvalue,
                                               const double* n_fn, int reversion, const double* h,
                                               const double* g, double* A, long long lda,
                                               double* b) {
  MFB_ARG(n_el_nodes > 0 && n_el_nodes <= 9 && rows && cols && ctype && cvalue && n_fn && h && g &&
              A && b && lda > 0,
          "invalid scatter arguments");
  const int rc = scatter_tables<double>(n_el_nodes, rows, cols, ctype, cvalue, n_fn, reversion, h,
                                        g, A, lda, b, false);
  if (rc) set_error("scatter: ctype must be 0, 1 or 10 with the matching columns present");
  return rc;
}

extern "C" int mfb_scatter_bem_harela_equation(int n_el_nodes, const int* rows, const int* cols,
                                               const int* ctype, const double* cvalue,
                                               const double* n_fn, int reversion, const double* h,
                                               const double* g, const double* u_inc,
                                               const double* t_inc, double* A, long long lda,
                                               double* b) {
  MFB_ARG(n_el_nodes > 0 && n_el_nodes <= 9 && rows && cols && ctype && cvalue && n_fn && h && g &&
              A && b && lda > 0 && (!u_inc) == (!t_inc),
          "invalid scatter arguments");
  typedef std::complex<double> z;
  const int rc = scatter_tables<z>(n_el_nodes, rows, cols, ctype, (const z*)cvalue, n_fn, reversion,
                                   (const z*)h, (const z*)g, (z*)A, lda, (z*)b, true);
  if (rc) {
    set_error("scatter: ctype must be 0, 1, 2, 3 or 10 with the matching columns present");
    return rc;
  }
  // incident wave field of the region (src/assemble_bem_harela_equation.f90:651-666):
  // b += h u_inc - g t_inc, u_inc / t_inc (3 x n_el_nodes) at the element's nodes
  if (u_inc) {
    const int ne = n_el_nodes;
    const z *H = (const z*)h, *G = (const z*)g, *U = (const z*)u_inc, *T = (const z*)t_inc;
    z* B = (z*)b;
    for (int il = 0; il < 3; il++)
      for (int ik = 0; ik < 3; ik++)
        for (int kn = 0; kn < ne; kn++) {
          const int o = kn + ne * il + 3 * ne * ik;
          B[rows[il]] += H[o] * U[ik + 3 * kn] - G[o] * T[ik + 3 * kn];
        }
  }
  return MFB_OK;
}

// Kernel blocks of independent (element, collocation point) pairs through the same kernels as the
// assembly: the GPU counterpart of fbem_bem_staela3d_sbie_auto / fbem_bem_harela3d_sbie_auto
// (bem_staela3d.f90:524-589, bem_harela3d.f90:1474-1538) for a batch of pairs.
static int pair_blocks(int npairs, const double* X, const double* xc, double qsi_re, int ns,
                       int n_ps, const int* ps_gln, int* classes, double* h, double* g,
                       bool harmonic, const KernelParams& kp) {
  MFB_ARG(npairs > 0 && X && xc && ps_gln && h && g, "null argument");
  // one element per pair (its own nodes) and one collocation point per pair; only the designated
  // pairs (element p, point p) are classified and integrated
  const int nn = 9 * npairs, ne = npairs;
  std::vector<double> x(3LL * nn);
  std::vector<int> conn(9LL * ne), ctype(3LL * nn, 1);
  std::vector<double> cval(3LL * nn, 0.0);
  CollocSet cs;
  cs.ncp = npairs;
  for (int p = 0; p < npairs; p++) {
    for (int k = 0; k < 9; k++) {
      conn[9 * p + k] = 9 * p + k;
      for (int c = 0; c < 3; c++) x[3 * (9 * p + k) + c] = X[27LL * p + 3 * k + c];
    }
    for (int c = 0; c < 3; c++) cs.xc.push_back(xc[3LL * p + c]);
    cs.cxi.push_back(0.0);
    cs.cxi.push_back(0.0);
    cs.crow.push_back(0);
    cs.cel.push_back(-1);
  }
  mfb_mesh_t m = nullptr;
  int rc = mesh_create_impl(nn, ne, x.data(), conn.data(), ctype.data(), cval.data(), qsi_re, ns,
                            n_ps, ps_gln, 1e-6, &cs, 0.0, false, &m);
  if (rc) return rc;
  std::vector<int> pids(npairs);
  for (int p = 0; p < npairs; p++) pids[p] = p * npairs + p;
  std::vector<unsigned char> cls(npairs);
  int* dp = nullptr;
  unsigned char* dc = nullptr;
  double* dblk = nullptr;
  const int w = harmonic ? 2 : 1;
  auto done = [&](int code) {
    (void)hipFree(dp);
    (void)hipFree(dc);
    (void)hipFree(dblk);
    mfb_mesh_destroy(m);
    return code;
  };
  hipError_t he = hipMalloc(&dp, sizeof(int) * npairs);
  if (he == hipSuccess) he = hipMalloc(&dc, npairs);
  if (he == hipSuccess) he = hipMemcpy(dp, pids.data(), sizeof(int) * npairs, hipMemcpyHostToDevice);
  if (he == hipSuccess) {
    hipLaunchKernelGGL(k_classify_listed, dim3((npairs + 127) / 128), dim3(128), 0, 0, m->dm,
                       m->d_qsp, dp, npairs, dc);
    he = hipGetLastError();
  }
  if (he == hipSuccess) he = hipMemcpy(cls.data(), dc, npairs, hipMemcpyDeviceToHost);
  if (he != hipSuccess) {
    set_error("pair_blocks: %s", hipGetErrorString(he));
    return done(MFB_ERR_HIP);
  }
  std::vector<std::vector<int>> lst(m->n_cls);
  for (int p = 0; p < npairs; p++) {
    classes[p] = cls[p];
    lst[cls[p]].push_back(pids[p]);
  }
  std::vector<int> flat;
  for (int c = 0; c < m->n_cls; c++) {
    m->cls_off[c] = (long long)flat.size();
    m->cls_cnt[c] = (long long)lst[c].size();
    flat.insert(flat.end(), lst[c].begin(), lst[c].end());
  }
  m->cls_off[m->n_cls] = (long long)flat.size();
  he = hipMalloc(&m->lists, sizeof(int) * flat.size());
  if (he == hipSuccess)
    he = hipMemcpy(m->lists, flat.data(), sizeof(int) * flat.size(), hipMemcpyHostToDevice);
  if (he == hipSuccess) he = hipMalloc((void**)&dblk, sizeof(double) * 162 * w * npairs);
  if (he != hipSuccess) {
    set_error("pair_blocks: %s", hipGetErrorString(he));
    return done(MFB_ERR_HIP);
  }
  rc = make_pair_geom(m);
  if (rc) return done(rc);
  rc = harmonic ? assemble<true>(m, kp, 0.0, nullptr, 0, nullptr, nullptr, dblk)
                : assemble<false>(m, kp, 0.0, nullptr, 0, nullptr, nullptr, dblk);
  if (rc == MFB_OK) {
    std::vector<double> hb(162LL * w * npairs);
    he = hipMemcpy(hb.data(), dblk, sizeof(double) * hb.size(), hipMemcpyDeviceToHost);
    if (he != hipSuccess) {
      set_error("pair_blocks: %s", hipGetErrorString(he));
      rc = MFB_ERR_HIP;
    }
    // blocks are in list order: slot q holds the pair of element flat[q] / npairs
    for (size_t q = 0; q < flat.size() && rc == MFB_OK; q++) {
      const long long p = flat[q] / npairs;
      for (int o = 0; o < 81 * w; o++) {
        h[81LL * w * p + o] = hb[162LL * w * q + o];
        g[81LL * w * p + o] = hb[162LL * w * q + 81 * w + o];
      }
    }
  }
  return done(rc);
}

extern "C" int mfb_pair_blocks_staela(int npairs, const double* X, const double* x_i, double mu,
                                      double nu, double qsi_relative_error, int qsi_ns_max,
                                      int n_precalsets, const int* precalset_gln, int* classes,
                                      double* h, double* g) {
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.cteu1 = 1.0 / (16.0 * kPi * mu * (1.0 - nu));
  kp.cteu2 = 3.0 - 4.0 * nu;
  kp.ctet1 = -1.0 / (8.0 * kPi * (1.0 - nu));
  kp.ctet2 = 1.0 - 2.0 * nu;
  return pair_blocks(npairs, X, x_i, qsi_relative_error, qsi_ns_max, n_precalsets, precalset_gln,
                     classes, h, g, false, kp);
}

extern "C" int mfb_pair_blocks_harela(int npairs, const double* X, const double* x_i, double omega,
                                      double lambda_re, double lambda_im, double mu_re,
                                      double mu_im, double rho, double qsi_relative_error,
                                      int qsi_ns_max, int n_precalsets, const int* precalset_gln,
                                      int* classes, double* h, double* g) {
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.harmonic = 1;
  host_har_params(lambda_re, lambda_im, mu_re, mu_im, rho, omega, &kp.h);
  return pair_blocks(npairs, X, x_i, qsi_relative_error, qsi_ns_max, n_precalsets, precalset_gln,
                     classes, h, g, true, kp);
}

// ------------------------------------------------------------------------------------------------
// interior points (src/calculate_internal_points_mechanics_static.f90,
// src/calculate_internal_points_mechanics_bem_harela.f90)
// ------------------------------------------------------------------------------------------------
struct mfb_points_s {
  mfb_mesh_t pm = nullptr;  // the boundary's elements with the points as collocation points
  int npts = 0;
};

// A point that coincides with a boundary node (distance below 1e-12 of the characteristic length
// of the node's first element) takes the node's displacement, as the reference does
// (src/calculate_internal_points_mechanics_bem_harela.f90:197-210).
// (found when the set is made: blockIdx.y runs over parts of the nodes; of several the last one)
__global__ void __launch_bounds__(128) k_snap_find(DevMesh m, int* snap) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= m.ncp) return;
  const double* xp = m.xc + 3 * p;
  int found = -1;
  for (int i = blockIdx.y; i < m.nn; i += gridDim.y) {
    if (m.inc_ptr[i + 1] == m.inc_ptr[i]) continue;
    const double cl = m.elem[8 * m.inc_e[m.inc_ptr[i]]];
    const double dx = xp[0] - m.x[3 * i], dy = xp[1] - m.x[3 * i + 1], dz = xp[2] - m.x[3 * i + 2];
    if (sqrt(dx * dx + dy * dy + dz * dz) / cl < 1e-12) found = i;
  }
  if (found >= 0) atomicMax(&snap[p], found);
}

template <typename T>
__global__ void k_snap_nodes(DevMesh m, const int* __restrict__ snap, const T* ub, T* out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= m.ncp || snap[p] < 0) return;
  for (int k = 0; k < 3; k++) out[3 * p + k] = ub[3 * snap[p] + k];
}

// the points in Morton order of a 1024^3 grid over their bounding box
static std::vector<int> morton_order(int n, const double* x) {
  double lo[3], hi[3];
  for (int c = 0; c < 3; c++) {
    lo[c] = hi[c] = x[c];
    for (int i = 1; i < n; i++) {
      lo[c] = std::min(lo[c], x[3LL * i + c]);
      hi[c] = std::max(hi[c], x[3LL * i + c]);
    }
  }
  const double side = std::max(std::max(hi[0] - lo[0], hi[1] - lo[1]), hi[2] - lo[2]);
  const double f = side > 0 ? 1023.0 / side : 0.0;
  std::vector<std::pair<unsigned, int>> key(n);
  for (int i = 0; i < n; i++) {
    unsigned k = 0;
    for (int c = 0; c < 3; c++) {
      const double t = (x[3LL * i + c] - lo[c]) * f;
      const unsigned v = t > 0 ? (unsigned)std::min(t, 1023.0) : 0u;   // (NaN: 0)
      for (int b = 0; b < 10; b++) k |= (v >> b & 1u) << (3 * b + c);
    }
    key[i] = {k, i};
  }
  std::sort(key.begin(), key.end());
  std::vector<int> o(n);
  for (int i = 0; i < n; i++) o[i] = key[i].second;
  return o;
}

extern "C" int mfb_points_create(mfb_mesh_t mesh, int npts, const double* x, mfb_points_t* out) {
  MFB_ARG(mesh && npts > 0 && x && out, "bad argument");
  CollocSet cs;
  cs.ncp = npts;
  cs.xc.assign(x, x + 3LL * npts);
  cs.cxi.assign(2LL * npts, 0.0);
  cs.crow.assign(npts, 0);
  cs.cel.assign(npts, -1);
  const DevMesh& d = mesh->dm;
  mfb_mesh_t pm = nullptr;
  int rc = mesh_create_impl(d.nn, d.ne, mesh->h_x.data(), mesh->h_conn.data(),
                            mesh->h_ctype.data(), mesh->h_cval.data(), d.qsi_re, d.ns_max, d.n_ps,
                            mesh->h_ps.data(), mesh->h_tol, &cs, 0.0, true, &pm);
  if (rc) return rc;
  const std::vector<int> order = morton_order(npts, x);
  hipError_t he = hipMalloc((void**)&pm->order, sizeof(int) * (size_t)npts);
  if (he == hipSuccess) he = hipMalloc((void**)&pm->snap, sizeof(int) * (size_t)npts);
  if (he == hipSuccess)
    he = hipMemcpy(pm->order, order.data(), sizeof(int) * (size_t)npts, hipMemcpyHostToDevice);
  if (he == hipSuccess) {
    hipLaunchKernelGGL(k_fill_int, dim3((npts + 255) / 256), dim3(256), 0, 0, pm->snap, npts, -1);
    hipLaunchKernelGGL(k_snap_find, dim3((npts + 127) / 128, std::min(64, d.nn)), dim3(128), 0, 0,
                       pm->dm, pm->snap);
    he = hipGetLastError();
  }
  if (he == hipSuccess) he = hipStreamSynchronize(0);
  if (he != hipSuccess) {
    mfb_mesh_destroy(pm);
    set_error("mfb_points_create: %s", hipGetErrorString(he));
    return MFB_ERR_HIP;
  }
  mfb_points_s* p = new mfb_points_s();
  p->pm = pm;
  p->npts = npts;
  *out = p;
  return MFB_OK;
}

extern "C" int mfb_points_destroy(mfb_points_t p) {
  if (!p) return MFB_OK;
  mfb_mesh_destroy(p->pm);
  delete p;
  return MFB_OK;
}

extern "C" int mfb_points_stats(mfb_points_t p, mfb_assembly_stats* st) {
  MFB_ARG(p, "null argument");
  return mfb_mesh_stats(p->pm, st);
}

extern "C" int mfb_points_pair_classes(mfb_points_t p, unsigned char* classes) {
  MFB_ARG(p, "null argument");
  return mfb_mesh_pair_classes(p->pm, classes);
}

template <bool H>
static int points_eval(mfb_points_t p, const KernelParams& kp, const double* ub, const double* tb,
                       double* out, void* stream) {
  typedef typename Val<H>::T T;
  MFB_ARG(p && ub && tb && out, "null argument");
  VecOut<T> v{(const T*)ub, (const T*)tb, (T*)out};
  int rc = assemble<H>(p->pm, kp, 0.0, nullptr, 0, nullptr, stream, nullptr, 0.0, v);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_snap_nodes<T>, dim3((p->npts + 127) / 128), dim3(128), 0, s, p->pm->dm,
                     p->pm->snap, (const T*)ub, (T*)out);
  MFB_HIP(hipGetLastError());
  MFB_HIP(hipStreamSynchronize(s));
  return MFB_OK;
}

extern "C" int mfb_points_displacement_staela(mfb_points_t p, double mu, double nu,
                                              const double* u_bnd, const double* t_bnd,
                                              double* u_out, void* stream) {
  MFB_ARG(mu > 0 && nu < 0.5 && nu > -1.0, "invalid elastic constants");
  return points_eval<false>(p, static_params(mu, nu), u_bnd, t_bnd, u_out, stream);
}

extern "C" int mfb_points_displacement_harela(mfb_points_t p, double omega, double lambda_re,
                                              double lambda_im, double mu_re, double mu_im,
                                              double rho, const double* u_bnd,
                                              const double* t_bnd, double* u_out, void* stream) {
  MFB_ARG(omega > 0 && rho > 0 && mu_re > 0, "invalid harmonic parameters (omega > 0 required)");
  KernelParams kp;
  std::memset(&kp, 0, sizeof kp);
  kp.harmonic = 1;
  host_har_params(lambda_re, lambda_im, mu_re, mu_im, rho, omega, &kp.h);
  return points_eval<true>(p, kp, u_bnd, t_bnd, u_out, stream);
}
