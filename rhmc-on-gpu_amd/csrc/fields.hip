// fields.hip -- gauge-field side of the RHMC molecular dynamics on gfx950:
// fermion force, gauge force, exp(i eps P) link update, momentum update,
// per-site action / Delta H, rational-function sums, RNG and the host-layout
// conversions of the C ABI.  All arithmetic here is FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <exception>
#include <thread>
#include <vector>

#include "context.hpp"

namespace rhmc {

static inline unsigned nblk(long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// --------------------------------------------------------------- fermion force
// fermionforce.cc:46-104 + ipdot.cc:83-155:
//   F_mu(e) =  sum_j a_j h_j(e+mu) (x) s_j(e)^*     (even sites)
//   F_mu(o) = -sum_j a_j s_j(o+mu) (x) h_j(o)^*     (odd sites)
//   ipdot_mu(x) = TA(U_mu(x) F_mu(x))   [+= existing ipdot if accumulate]
// s_j: shifted solutions (even), h_j = D_oe s_j (odd); one thread per site
// holds the four F_mu in registers (FP64) and reads each spinor of its site
// once.  C = double2 (FP64 solutions) or float2 (FP32 solutions of the FP32
// MD solves).
// One thread per site and system at a time: the 15 loads of a system
// (uniform base + 32-bit lane offset) are issued before its multiply-adds.
// Taking two systems per step keeps more loads in flight but needs ~280
// VGPRs (one wave per SIMD) and measured slower.  So did two lanes per site
// (two F_mu each, loads of system j+1 issued before system j's multiply-
// adds, 166 VGPRs): 522 against 415 us for 128 FP32 systems at 32^3x8 (both
// with the earlier parity-major grid).  The kernel is bound by load-
// instruction issue, and that split issues 18 loads per site and system
// instead of 15.
template <typename C, int NQ>
__device__ __forceinline__ void ff_systems(const C *own_v, const C *nb_v, long Vh, int j0, unsigned ho,
                                           const unsigned (&nbo)[4], const double *coef, double sgn,
                                           Mat<double> (&F)[4]) {
  C own[NQ][3], w[NQ][4][3];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const long base = (long)(j0 + q) * 3 * Vh;
#pragma unroll
    for (int k = 0; k < 3; k++) own[q][k] = ld_off(own_v + base + (long)k * Vh, ho);
#pragma unroll
    for (int mu = 0; mu < 4; mu++)
#pragma unroll
      for (int i = 0; i < 3; i++) w[q][mu][i] = ld_off(nb_v + base + (long)i * Vh, nbo[mu]);
  }
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const double a = sgn * coef[j0 + q];
    double2 o[3];
#pragma unroll
    for (int k = 0; k < 3; k++) o[k] = make_double2((double)own[q][k].x, -(double)own[q][k].y);  // conjugate
#pragma unroll
    for (int mu = 0; mu < 4; mu++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const double2 v = make_double2(a * (double)w[q][mu][i].x, a * (double)w[q][mu][i].y);
#pragma unroll
        for (int k = 0; k < 3; k++) cfma(F[mu].e[i][k], v, o[k]);
      }
  }
}

// Grid: both parities of each kBlock-site tile, consecutive on one XCD, the
// tiles in the XCD-compact order of the Dslash (tiles, or lattice order when
// null): the even sites read the odd spinors that the odd sites of the same
// tile read as their own, and the +mu neighbours stay in the XCD's share, so
// more of a spinor's five uses find it in that XCD's L2 (FP64, 128 systems
// at 32^3x8: 5.84 -> 4.36 GB fetched per call, 816 -> 648 us).
// U: the FP64 18-real links for FP64 solutions, the FP64 12-real copy for FP32
// ones (the links an MD with FP32 solves keeps).
template <typename C>
__global__ __launch_bounds__(kBlock) void k_fermion_force(LatticeDims L, const int *tiles, const double2 *U,
                                                          const C *s, const C *hv, const double *coef, int nsys,
                                                          double2 *ipdot, int accumulate) {
  const long Vh = L.Vh;
  const unsigned b = xcd_block(blockIdx.x, gridDim.x);
  const int par = (int)(b & 1u);
  const int q = (int)(b >> 1);
  const int h = (tiles ? tiles[q] : q) * kBlock + (int)threadIdx.x;
  if (h >= (int)Vh) return;
  const SiteCoord c = site_coords_i(L, par, h);
  unsigned nbo[4];
#pragma unroll
  for (int mu = 0; mu < 4; mu++) nbo[mu] = (unsigned)neighbour_i(L, c, mu, +1) * (unsigned)sizeof(C);
  const unsigned ho = (unsigned)h * (unsigned)sizeof(C);
  Mat<double> F[4];
#pragma unroll
  for (int mu = 0; mu < 4; mu++)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int k = 0; k < 3; k++) F[mu].e[i][k] = make_double2(0.0, 0.0);
  const C *own_v = par == 0 ? s : hv;
  const C *nb_v = par == 0 ? hv : s;
  const double sgn = par == 0 ? 1.0 : -1.0;
  for (int j = 0; j < nsys; j++) ff_systems<C, 1>(own_v, nb_v, Vh, j, ho, nbo, coef, sgn, F);
#pragma unroll
  for (int mu = 0; mu < 4; mu++) {
    Mat<double> Um;
    if constexpr (sizeof(C) == sizeof(double2)) Um = load_link_d18(U, Vh, mu, par, h);
    else Um = load_link_d12(U, Vh, mu, par, h, eta_phase(L, c.x, c.y, c.z, c.t, mu));
    Mat<double> T = ta(mmul(Um, F[mu]));
    if (accumulate) {
      const Mat<double> old = load_aherm(ipdot, Vh, mu, par, h);
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = 0; k < 3; k++) T.e[i][k] = cadd(T.e[i][k], old.e[i][k]);
    }
    store_aherm(ipdot, Vh, mu, par, h, T);
  }
}

// The force's coefficients in device memory: uploaded only when they differ
// from the ones the buffer already holds (every MD force of a trajectory
// uses the same ones), so the force launches follow the solve without a copy.
static bool force_coef_upload(Context &c, double *dcoef, const double *num, int nsys) {
  std::vector<double> &held = c.force_coef_held;
  if (c.force_coef_dev == dcoef && held.size() == (size_t)nsys && std::equal(held.begin(), held.end(), num))
    return true;
  c.force_coef_dev = nullptr;
  if (!h2d(c, dcoef, num, sizeof(double) * nsys)) return false;
  held.assign(num, num + nsys);
  c.force_coef_dev = dcoef;
  return true;
}

int fermion_force(Context &c, int nsys, const double *num, const double2 *x, int accumulate) {
  // nsys = n_pf * order systems, x = [n_pf][order][3][Vh]; num has nsys entries
  const long Vh = c.Vh;
  size_t need = sizeof(double2) * 3 * Vh * (size_t)nsys;
  // h_j = D_oe s_j for all systems (one multi-RHS hop sharing link loads),
  // into workspace buffers kept for the context's lifetime
  double2 *hv = (double2 *)scratch_get(c, SCR_FORCE_HOP, need);
  double *coef = (double *)scratch_get(c, SCR_FORCE_COEF, sizeof(double) * 256);
  if (!hv || !coef || nsys > 256) return -1;
  if (!force_coef_upload(c, coef, num, nsys)) return -1;
  launch_hop_d(c, 1, x, hv, nsys, 3 * Vh, 3 * Vh);
  hipLaunchKernelGGL(k_fermion_force<double2>, dim3(2 * nblk(Vh)), dim3(kBlock), 0, c.stream, c.L, c.tiles, c.U64, x, hv, coef,
                     nsys, c.ipdot, accumulate);
  // stream-ordered for the caller (the coefficients are staged in pinned memory)
  return hip_ok(c, hipGetLastError(), "fermion force") ? 0 : -1;
}

int fermion_force32(Context &c, int nsys, const double *num, const float2 *x32, int accumulate) {
  const long Vh = c.Vh;
  float2 *hv = (float2 *)scratch_get(c, SCR_FORCE_HOP, sizeof(float2) * 3 * Vh * (size_t)nsys);
  double *coef = (double *)scratch_get(c, SCR_FORCE_COEF, sizeof(double) * 256);
  if (!hv || !coef || nsys > 256) return -1;
  if (!force_coef_upload(c, coef, num, nsys)) return -1;
  launch_hop_s(c, 1, x32, hv, nsys, 3 * Vh, 3 * Vh);
  hipLaunchKernelGGL(k_fermion_force<float2>, dim3(2 * nblk(Vh)), dim3(kBlock), 0, c.stream, c.L, c.tiles, c.U64c, x32, hv, coef,
                     nsys, c.ipdot, accumulate);
  // stream-ordered for the caller (the coefficients are staged in pinned memory)
  return hip_ok(c, hipGetLastError(), "fermion force") ? 0 : -1;
}

// ------------------------------------------------ allocation-free fermion force
// For callers that cannot allocate device memory (graph capture, tight
// serving loops): the force's scratch -- the coefficients and the hop
// results h_j = D_oe s_j -- lives in one fixed file-scope device array.
// Every GPU holds its own copy of it until the process ends.  In host code
// the name `scratch` is only a stand-in for the symbol: kernels are given
// the per-device address that hipGetSymbolAddress returned.
constexpr size_t kNoAllocCoefBytes = 256 * sizeof(double);  // 2 KiB, keeps h 256-byte aligned
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDeviceOrdinal = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDeviceOrdinal];

int noalloc_scratch_init(Context &c) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  c.noalloc_scratch = nullptr;
  if (c.device < 0 || c.device >= kMaxDeviceOrdinal) return -1;
  if (!g_scratch_ptr[c.device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return -1;
    }
    g_scratch_ptr[c.device] = p;
  }
  c.noalloc_scratch = g_scratch_ptr[c.device];
  return 0;
}

// the coefficients travel by value in the kernel arguments, so nothing is
// staged through host memory
struct CoefTable {
  double v[256];
};
__global__ void k_coef_store(CoefTable t, int n, double *dst) {
  const int i = threadIdx.x;
  if (i < n) dst[i] = t.v[i];
}

int fermion_force_noalloc(Context &c, int order, const double *num, int accumulate) {
  const long Vh = c.Vh;
  const int nsys = c.n_pf * order;
  const size_t per_sys = sizeof(double2) * 3 * (size_t)Vh;
  const size_t room = kNoAllocScratchBytes - kNoAllocCoefBytes;
  if (per_sys > room) {
    c.last_error = "gpu_fermion_force_noalloc: one system (48 V/2 bytes) exceeds the 64 MiB fixed scratch";
    return -2;
  }
  if (!c.noalloc_scratch) {
    c.last_error = "gpu_fermion_force_noalloc: device address of the fixed scratch unavailable";
    return -1;
  }
  if (nsys < 1 || nsys > 256) return -2;
  CoefTable t;
  for (int j = 0; j < nsys; j++) t.v[j] = num[j % order];  // system j = ps * order + k
  double *coef = (double *)c.noalloc_scratch;
  double2 *hv = (double2 *)((unsigned char *)c.noalloc_scratch + kNoAllocCoefBytes);
  hipLaunchKernelGGL(k_coef_store, dim3(1), dim3(256), 0, c.stream, t, nsys, coef);
  // groups of systems whose hop results fit the scratch; the force of each
  // group is added to the previous groups' (TA and U F are linear)
  const int group = (int)std::min<size_t>((size_t)nsys, room / per_sys);
  for (int j0 = 0; j0 < nsys; j0 += group) {
    const int n = std::min(group, nsys - j0);
    const double2 *x = c.smf + (long)j0 * 3 * Vh;
    launch_hop_d_fixed(c, 1, x, hv, n, 3 * Vh, 3 * Vh);
    hipLaunchKernelGGL(k_fermion_force<double2>, dim3(2 * nblk(Vh)), dim3(kBlock), 0, c.stream, c.L, c.tiles, c.U64, x, hv,
                       coef + j0, n, c.ipdot, (j0 > 0 || accumulate) ? 1 : 0);
  }
  return hip_ok(c, hipGetLastError(), "fermion force (fixed scratch)") ? 0 : -1;
}

// ----------------------------------------------------------------- gauge force
// staples.cc:16-74, ipdot.cc:25-79:
//   ipdot_mu(x) = TA(U_mu(x) beta/3 sum_{nu!=mu} [U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
//                                              + U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)])
// Links come from the FP64 12-real copy.  A staple is a product of three links,
// each unitary with a known sign (its staggered phase), so it is unitary with
// the product of the signs, and only its first two rows are multiplied out;
// the third is rebuilt once from them, as it is for the links that are needed
// whole: 369 complex products per link instead of 465.
struct Rows {
  double2 e[2][3];
};
// rows 0 and 1 of link mu at half index h of parity par
__device__ __forceinline__ void rows_load(const double2 *U12, long Vh, int mu, int par, int h, Rows &m) {
  const double2 *b = U12 + (long)(mu * 2 + par) * 6 * Vh;
  const unsigned off = (unsigned)h * (unsigned)sizeof(double2);
#pragma unroll
  for (int k = 0; k < 6; k++) m.e[k / 3][k % 3] = ld_off(b + (long)k * Vh, off);
}
// the whole matrix, its sign (-1 for an odd number of phases) on row 2
__device__ __forceinline__ Mat<double> rows_mat(const Rows &r, int odd) {
  Mat<double> m;
#pragma unroll
  for (int k = 0; k < 6; k++) m.e[k / 3][k % 3] = r.e[k / 3][k % 3];
  rebuild_row2(m, odd & 1 ? -1.0 : 1.0);
  return m;
}
// rows of a b^+ and of a b
__device__ __forceinline__ Rows rows_nd(const Rows &a, const Mat<double> &b) {
  Rows r;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) {
      double2 s = cmul(a.e[i][0], cconj(b.e[j][0]));
      cfma(s, a.e[i][1], cconj(b.e[j][1]));
      cfma(s, a.e[i][2], cconj(b.e[j][2]));
      r.e[i][j] = s;
    }
  return r;
}
__device__ __forceinline__ Rows rows_nn(const Rows &a, const Mat<double> &b) {
  Rows r;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) {
      double2 s = cmul(a.e[i][0], b.e[0][j]);
      cfma(s, a.e[i][1], b.e[1][j]);
      cfma(s, a.e[i][2], b.e[2][j]);
      r.e[i][j] = s;
    }
  return r;
}
// Ends a stage: the values pass through an empty asm statement (in-out
// operands, memory clobber), so the stage's multiply-adds are issued after
// the loads before it in program order and before those that follow.
__device__ __forceinline__ void rows_fence(Rows &r) {
#pragma unroll
  for (int k = 0; k < 6; k++) asm volatile("" : "+v"(r.e[k / 3][k % 3].x), "+v"(r.e[k / 3][k % 3].y) : : "memory");
}
__device__ __forceinline__ void mat_fence(Mat<double> &m) {
#pragma unroll
  for (int k = 0; k < 9; k++) asm volatile("" : "+v"(m.e[k / 3][k % 3].x), "+v"(m.e[k / 3][k % 3].y) : : "memory");
}
__device__ __forceinline__ void rows_add(Mat<double> &st, const Rows &r, int odd) {
  const Mat<double> m = rows_mat(r, odd);
#pragma unroll
  for (int k = 0; k < 9; k++) st.e[k / 3][k % 3] = cadd(st.e[k / 3][k % 3], m.e[k / 3][k % 3]);
}

// P += i step F at one link (momenta.cc:82-115): the force it has just formed
__device__ __forceinline__ void mom_add(double2 *P, long Vh, int mu, int par, int h, const Mat<double> &F, double s) {
  double2 *b = P + (long)(mu * 2 + par) * 4 * Vh + h;
  const double2 f[3] = {F.e[0][1], F.e[0][2], F.e[1][2]};
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double2 p = b[(long)k * Vh];
    p.x -= s * f[k].y;
    p.y += s * f[k].x;
    b[(long)k * Vh] = p;
  }
  double2 d = b[3 * Vh];
  d.x -= s * F.e[0][0].y;
  d.y -= s * F.e[1][1].y;
  b[3 * Vh] = d;
}

// number of phases (mod 2) of the link (c, MU); dt: c.t moved by that much
template <int MU>
__device__ __forceinline__ int phases(const LatticeDims &L, const SiteCoord &c, int dt = 0) {
  if (MU == 0) return 0;
  if (MU == 1) return c.x;
  if (MU == 2) return c.x + c.y;
  const int t = dt < 0 ? (c.t == 0 ? L.nt - 1 : c.t - 1) : c.t;
  return c.x + c.y + c.z + (L.antiperiodic_t && t == L.nt - 1 ? 1 : 0);
}

// The staples of link (c, MU) in the plane with the N-th other direction,
// added to st; la, lb hold the first two links (U_nu(x+mu), U_mu(x+nu)) on
// entry and those of the next plane on return.  df, db: change of the half
// index one step forward and backward (the index is a sum of one term per
// coordinate, so two steps add up).
template <int MU, int N>
__device__ __forceinline__ void plane_loads(const double2 *U12, const LatticeDims &L, int par, int h,
                                            const int (&df)[4], Rows &la, Rows &lb) {
  constexpr int NU = N < MU ? N : N + 1;
  rows_load(U12, L.Vh, NU, 1 - par, h + df[MU], la);
  rows_load(U12, L.Vh, MU, 1 - par, h + df[NU], lb);
}
template <int MU, int N>
__device__ __forceinline__ void plane_staples(const double2 *U12, const LatticeDims &L, int par, const SiteCoord &c,
                                              int h, const int (&df)[4], const int (&db)[4], Rows &la, Rows &lb,
                                              Mat<double> &st) {
  constexpr int NU = N < MU ? N : N + 1;
  const long Vh = L.Vh;
  // phases: a step along d changes those of direction e > d
  const int pn = phases<NU>(L, c), pm = phases<MU>(L, c);
  const int n_at_mu = pn + (MU < NU), m_at_nu = pm + (NU < MU);  // U_nu(x+-mu), U_mu(x+-nu)
  const int back = phases<NU>(L, c, -1);                         // U_nu(x-nu)
  // upper: U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
  Rows l3, a;
  rows_load(U12, Vh, NU, par, h, l3);
  a = rows_nd(la, rows_mat(lb, m_at_nu));
  rows_fence(a);
  Rows l4, l5;
  rows_load(U12, Vh, NU, par, h + df[MU] + db[NU], l4);
  rows_load(U12, Vh, MU, 1 - par, h + db[NU], l5);
  a = rows_nd(a, rows_mat(l3, pn));
  rows_add(st, a, n_at_mu + m_at_nu + pn);
  mat_fence(st);
  // lower: U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)
  Rows l6;
  rows_load(U12, Vh, NU, 1 - par, h + db[NU], l6);
  const int n4 = back + (MU < NU);
  {
    const Mat<double> m = rows_mat(l4, n4);
    Rows d;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int k = 0; k < 3; k++) d.e[i][k] = cconj(m.e[k][i]);
    a = rows_nd(d, rows_mat(l5, m_at_nu));
  }
  rows_fence(a);
  if constexpr (N < 2) plane_loads<MU, N + 1>(U12, L, par, h, df, la, lb);
  else rows_load(U12, Vh, MU, par, h, la);  // U_mu(x) for the last product
  a = rows_nn(a, rows_mat(l6, back));
  rows_add(st, a, n4 + m_at_nu + back);
  mat_fence(st);
}

template <int MU>
__device__ __forceinline__ void gauge_force_link(const LatticeDims &L, const double2 *U12, double b3, double2 *ipdot,
                                                 int accumulate, double2 *P, double step, int par, int h) {
  const long Vh = L.Vh;
  const SiteCoord c = site_coords_i(L, par, h);
  int df[4], db[4];
#pragma unroll
  for (int d = 0; d < 4; d++) {
    df[d] = neighbour_i(L, c, d, +1) - h;
    db[d] = neighbour_i(L, c, d, -1) - h;
  }
  Mat<double> st;
#pragma unroll
  for (int k = 0; k < 9; k++) st.e[k / 3][k % 3] = make_double2(0.0, 0.0);
  Rows la, lb;
  plane_loads<MU, 0>(U12, L, par, h, df, la, lb);
  plane_staples<MU, 0>(U12, L, par, c, h, df, db, la, lb, st);
  plane_staples<MU, 1>(U12, L, par, c, h, df, db, la, lb, st);
  plane_staples<MU, 2>(U12, L, par, c, h, df, db, la, lb, st);
  Mat<double> T = mmul(rows_mat(la, phases<MU>(L, c)), st);
#pragma unroll
  for (int k = 0; k < 9; k++) T.e[k / 3][k % 3] = cscale(T.e[k / 3][k % 3], b3);
  T = ta(T);
  if (accumulate) {
    const Mat<double> old = load_aherm(ipdot, Vh, MU, par, h);
#pragma unroll
    for (int k = 0; k < 9; k++) T.e[k / 3][k % 3] = cadd(T.e[k / 3][k % 3], old.e[k / 3][k % 3]);
  }
  store_aherm(ipdot, Vh, MU, par, h, T);
  if (P) mom_add(P, Vh, MU, par, h, T, step);
}

// staples.cc:16-74 + ipdot.cc:25-79: ipdot_mu(x) = TA(U_mu(x) beta/3 sum_nu
// [U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+ + U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)]).
// One link per lane, 19 link loads of 96 bytes, the links of each product
// loaded during the product before it: 206 VGPRs, two waves per SIMD (three,
// with 8 registers spilled, run the same).  32^3x8: 118 us per call (a form
// that multiplied whole matrices and hoisted all loads, one wave per SIMD,
// took 174); its FP64 multiply-adds alone are 42 us, its loads through L1
// 49 us, its 168 MB 35 us.
// Grid: the eight (parity, mu) workgroups of each kBlock-site tile
// consecutive on one XCD, the tiles in the XCD-compact order of the Dslash
// (tiles, or lattice order when null), so the links a tile's staples share
// are fetched into that XCD's L2 together.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_gauge_force(
    LatticeDims L, const int *tiles, const double2 *U12, double b3, double2 *ipdot, int accumulate, double2 *P,
    double step) {
  const unsigned b = xcd_block(blockIdx.x, gridDim.x);
  const int mu = (int)(b & 3u);
  const int par = (int)((b >> 2) & 1u);
  const int q = (int)(b >> 3);
  const int h = (tiles ? tiles[q] : q) * kBlock + (int)threadIdx.x;
  if (h >= (int)L.Vh) return;
  switch (mu) {
    case 0: gauge_force_link<0>(L, U12, b3, ipdot, accumulate, P, step, par, h); break;
    case 1: gauge_force_link<1>(L, U12, b3, ipdot, accumulate, P, step, par, h); break;
    case 2: gauge_force_link<2>(L, U12, b3, ipdot, accumulate, P, step, par, h); break;
    default: gauge_force_link<3>(L, U12, b3, ipdot, accumulate, P, step, par, h); break;
  }
}

int gauge_force(Context &c, int accumulate) {
  hipLaunchKernelGGL(k_gauge_force, dim3(8 * nblk(c.Vh)), dim3(kBlock), 0, c.stream, c.L, c.tiles, c.U64c,
                     c.beta / 3.0, c.ipdot, accumulate, (double2 *)nullptr, 0.0);
  return hip_ok(c, hipGetLastError(), "gauge force") ? 0 : -1;
}

// the gauge force and the momentum update with it (gauge_force, then
// momenta_update) in one pass
int gauge_kick(Context &c, int accumulate, double step) {
  hipLaunchKernelGGL(k_gauge_force, dim3(8 * nblk(c.Vh)), dim3(kBlock), 0, c.stream, c.L, c.tiles, c.U64c,
                     c.beta / 3.0, c.ipdot, accumulate, c.P, step);
  return hip_ok(c, hipGetLastError(), "gauge kick") ? 0 : -1;
}

// ------------------------------------------------------------ link update
// momenta.cc:42-78 + su3.cc:187-219 + conf.cc:235-251:
//   U <- Pi_SU3[ exp6(i step P) ] U, then Gram-Schmidt and row 2 *= eta.
// Writes the FP64 12-real copy and, when given, the 18-real links and the
// FP32 copy; reads the 18-real links, or the 12-real copy when they are stale
// (from12).
__global__ __launch_bounds__(kBlock) void k_exp_update(LatticeDims L, const double2 *P, double step, const double2 *Uin,
                                                       int from12, double2 *U, float4 *U32, double2 *U64c) {
  const long Vh = L.Vh;
  const int bx = xcd_block(blockIdx.x, gridDim.x);
  const long h = (long)bx * kBlock + threadIdx.x;
  const int par = blockIdx.y, mu = blockIdx.z;
  if (h >= Vh) return;
  const Mat<double> Pm = load_herm(P, Vh, mu, par, h);
  Mat<double> X;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int k = 0; k < 3; k++) X.e[i][k] = make_double2(-step * Pm.e[i][k].y, step * Pm.e[i][k].x);
  Mat<double> E, A = X;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int k = 0; k < 3; k++) E.e[i][k] = make_double2((i == k) ? 1.0 : 0.0, 0.0);
  const double cf[6] = {1.0, 0.5, 1.0 / 3.0, 0.25, 0.2, 1.0 / 6.0};
#pragma unroll
  for (int n = 0; n < 6; n++) {
    if (n > 0) {
      A = mmul(A, X);
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = 0; k < 3; k++) A.e[i][k] = cscale(A.e[i][k], cf[n]);
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int k = 0; k < 3; k++) E.e[i][k] = cadd(E.e[i][k], A.e[i][k]);
  }
  sunitarize(E);
  const SiteCoord c = site_coords_i(L, par, (int)h);
  const double eta = eta_phase(L, c.x, c.y, c.z, c.t, mu);
  Mat<double> Un = mmul(E, from12 ? load_link_d12(Uin, Vh, mu, par, h, eta) : load_link_d18(Uin, Vh, mu, par, h));
  sunitarize(Un);
#pragma unroll
  for (int k = 0; k < 3; k++) Un.e[2][k] = cscale(Un.e[2][k], eta);
  if (U) store_link_d18(U, Vh, mu, par, h, Un);
  if (U32) store_link_s12(U32, Vh, mu, par, h, Un);
  store_link_d12(U64c, Vh, mu, par, h, Un);
}

// 18-real links and FP32 copy of the FP64 12-real copy
__global__ __launch_bounds__(kBlock) void k_links_from12(LatticeDims L, const double2 *U64c, double2 *U, float4 *U32) {
  const long Vh = L.Vh;
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int par = blockIdx.y, mu = blockIdx.z;
  if (h >= Vh) return;
  const SiteCoord c = site_coords_i(L, par, (int)h);
  const Mat<double> m = load_link_d12(U64c, Vh, mu, par, h, eta_phase(L, c.x, c.y, c.z, c.t, mu));
  store_link_d18(U, Vh, mu, par, h, m);
  store_link_s12(U32, Vh, mu, par, h, m);
}

// Inside an MD (keep below LINKS_ALL) only the copies its solves and forces
// read are written: 256 bytes per link instead of 496 for a quenched one (32^3x8:
// 85 -> 50 us per update), 304 with FP32 solves; links_complete then restores
// the others, once.
int exp_update(Context &c, double step, int keep) {
  const bool all = keep == LINKS_ALL;
  hipLaunchKernelGGL(k_exp_update, dim3(nblk(c.Vh), 2, 4), dim3(kBlock), 0, c.stream, c.L, c.P, step,
                     c.links_stale ? c.U64c : c.U64, c.links_stale ? 1 : 0, all ? c.U64 : nullptr,
                     keep >= LINKS_FP32 ? c.U32 : nullptr, c.U64c);
  c.links_stale = !all;
  return hip_ok(c, hipGetLastError(), "exp update") ? 0 : -1;
}

int links_complete(Context &c) {
  if (!c.links_stale) return 0;
  c.links_stale = false;
  hipLaunchKernelGGL(k_links_from12, dim3(nblk(c.Vh), 2, 4), dim3(kBlock), 0, c.stream, c.L, c.U64c, c.U64, c.U32);
  return hip_ok(c, hipGetLastError(), "links complete") ? 0 : -1;
}

__global__ __launch_bounds__(kBlock) void k_refresh32(LatticeDims L, const double2 *U, float4 *U32, double2 *U64c) {
  const long Vh = L.Vh;
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int par = blockIdx.y, mu = blockIdx.z;
  if (h >= Vh) return;
  const Mat<double> m = load_link_d18(U, Vh, mu, par, h);
  store_link_s12(U32, Vh, mu, par, h, m);
  store_link_d12(U64c, Vh, mu, par, h, m);
}

// the FP32 12-real and FP64 12-real copies of the FP64 links
int refresh_links32(Context &c) {
  hipLaunchKernelGGL(k_refresh32, dim3(nblk(c.Vh), 2, 4), dim3(kBlock), 0, c.stream, c.L, c.U64, c.U32, c.U64c);
  return hip_ok(c, hipGetLastError(), "refresh links32") ? 0 : -1;
}

// -------------------------------------------------------- momentum update
// momenta.cc:82-115: P <- P + (i step) ipdot on the packed 8-real fields
__global__ __launch_bounds__(kBlock) void k_mom_update(double2 *P, const double2 *A, double s, long Vh, long n) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int slot = (int)((i / Vh) & 3);
  double2 p = P[i];
  const double2 a = A[i];
  if (slot < 3) {
    p.x -= s * a.y;
    p.y += s * a.x;
  } else {
    p.x -= s * a.x;
    p.y -= s * a.y;
  }
  P[i] = p;
}

int momenta_update(Context &c, double step) {
  const long n = 32 * c.Vh;
  hipLaunchKernelGGL(k_mom_update, dim3(nblk(n)), dim3(kBlock), 0, c.stream, c.P, c.ipdot, step, c.Vh, n);
  return hip_ok(c, hipGetLastError(), "momenta update") ? 0 : -1;
}

// P <- s P (revupdate.cc:53, reverse_momenta with s = -1)
__global__ __launch_bounds__(kBlock) void k_scale_inplace(double2 *v, double s, long n) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double2 p = v[i];
  v[i] = make_double2(s * p.x, s * p.y);
}

int momenta_scale(Context &c, double s) {
  const long n = 32 * c.Vh;
  hipLaunchKernelGGL(k_scale_inplace, dim3(nblk(n)), dim3(kBlock), 0, c.stream, c.P, s, n);
  return hip_ok(c, hipGetLastError(), "momenta scale") ? 0 : -1;
}

// ------------------------------------------------------------ solution sums
// rationalapprox.cc:269-369 / cuda_sol_sum: io[ps] = a0 io[ps] + sum_k a_k x[ps][k]
__global__ __launch_bounds__(kBlock) void k_sol_sum(double2 *io, const double2 *x, int nshift, double a0,
                                                    const double *num, long n3) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  const int ps = blockIdx.y;
  if (i >= n3) return;
  double2 v = io[(long)ps * n3 + i];
  v.x *= a0;
  v.y *= a0;
  for (int k = 0; k < nshift; k++) {
    const double2 xv = x[((long)ps * nshift + k) * n3 + i];
    v.x += num[k] * xv.x;
    v.y += num[k] * xv.y;
  }
  io[(long)ps * n3 + i] = v;
}

int sol_sum(Context &c, double2 *io, const double2 *x, int nshift, double a0, const double *num) {
  double *d = (double *)scratch_get(c, SCR_SOLSUM_COEF, sizeof(double) * kMaxShifts);
  if (!d || nshift > kMaxShifts) return -1;
  std::vector<double> h(num, num + nshift);
  if (!h2d(c, d, h.data(), sizeof(double) * nshift)) return -1;
  const long n3 = 3 * c.Vh;
  hipLaunchKernelGGL(k_sol_sum, dim3(nblk(n3), c.n_pf), dim3(kBlock), 0, c.stream, io, x, nshift, a0, d, n3);
  return hip_ok(c, hipStreamSynchronize(c.stream), "sol_sum") ? 0 : -1;
}

// ------------------------------------------------------------------- action
// Re tr of the plaquette (x; mu, nu) from the 18-real links: with A = U_mu(x)
// U_nu(x+mu) and B = U_nu(x) U_mu(x+nu) it is the real part of sum A_ij B_ij^*, two
// matrix products and nine complex ones instead of three products.  mu and
// nu are the same in a wave; one copy of the code for all planes (a kernel
// that runs once per measurement mostly waits for its instructions).
__device__ __forceinline__ double plaq_re(const LatticeDims &L, const double2 *U, int par, int h, const SiteCoord &c,
                                          int mu, int nu) {
  const long Vh = L.Vh;
  const int hm = neighbour_i(L, c, mu, +1), hn = neighbour_i(L, c, nu, +1);
  const Mat<double> a = mmul(load_link_d18(U, Vh, mu, par, h), load_link_d18(U, Vh, nu, 1 - par, hm));
  const Mat<double> b = mmul(load_link_d18(U, Vh, nu, par, h), load_link_d18(U, Vh, mu, 1 - par, hn));
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    s = fmar(a.e[k / 3][k % 3].x, b.e[k / 3][k % 3].x, s);
    s = fmar(a.e[k / 3][k % 3].y, b.e[k / 3][k % 3].y, s);
  }
  return s;
}

// action.cc:6-156: per-site contributions in the reference's order
//   init 0 : v  = sum_plaq beta/3 Re tr(plaq) + sum_mu 1/2 Re tr P^2 + sum_ps |phi|^2
//   init -1: v -= the same with Re<phi_new, chi> for the fermions
__global__ __launch_bounds__(kBlock) void k_action(LatticeDims L, const double2 *U, const double2 *P, double b3,
                                                   const double2 *phi, const double2 *chi, int npf, int with_f,
                                                   double *value, int init) {
  // both parities of a tile follow each other on one XCD, each XCD a part of
  // the lattice (32^3x8: 117 -> 89 us)
  const long Vh = L.Vh;
  const unsigned b = xcd_block(blockIdx.x, gridDim.x);
  const int par = (int)(b & 1u);
  const long h = (long)(b >> 1) * kBlock + threadIdx.x;
  if (h >= Vh) return;
  const long idx = (long)par * Vh + h;
  double v = init == 0 ? 0.0 : value[idx];
  const double sg = init == 0 ? 1.0 : -1.0;
  const SiteCoord c = site_coords_i(L, par, (int)h);
#pragma unroll 1
  for (int mu = 0; mu < 3; mu++)
#pragma unroll 1
    for (int nu = mu + 1; nu < 4; nu++) v += sg * b3 * plaq_re(L, U, par, (int)h, c, mu, nu);
  for (int mu = 0; mu < 4; mu++) {
    const Mat<double> pm = load_herm(P, Vh, mu, par, h);
    const Mat<double> q = mmul(pm, pm);
    v += sg * 0.5 * (q.e[0][0].x + q.e[1][1].x + q.e[2][2].x);
  }
  if (with_f && par == 0) {
    for (int ps = 0; ps < npf; ps++) {
      double f = 0.0;
      for (int k = 0; k < 3; k++) {
        const double2 a = phi[((long)ps * 3 + k) * Vh + h];
        const double2 b = init == 0 ? a : chi[((long)ps * 3 + k) * Vh + h];
        f += a.x * b.x + a.y * b.y;
      }
      v += sg * f;
    }
  }
  value[idx] = v;
}

int action_local(Context &c, const double2 *phi, const double2 *chi, int with_f, int init) {
  hipLaunchKernelGGL(k_action, dim3(2 * nblk(c.Vh)), dim3(kBlock), 0, c.stream, c.L, c.U64, c.P, c.beta / 3.0, phi,
                     chi, c.n_pf, with_f, c.action, init);
  return hip_ok(c, hipGetLastError(), "action") ? 0 : -1;
}

// include/tools.h:25-57 pairwise fold, same association order as the
// reference: n even, v[k] += v[k + n/2] for k < n/2; n odd, v[k] += v[k + n/2
// + 1] for k < n/2 and the middle value stays.  Array y of a launch starts at
// v + y stride.
__global__ __launch_bounds__(kBlock) void k_fold(double *v, long stride, long j, long off) {
  const long k = (long)blockIdx.x * kBlock + threadIdx.x;
  v += blockIdx.y * stride;
  if (k < j) v[k] += v[k + off];
}
// LV halvings at once: value k of n / 2^LV gathers the 2^LV values that the
// halvings add to it, in their order
template <int LV>
__global__ __launch_bounds__(kBlock) void k_fold_levels(double *v, long stride, long m) {
  const long k = (long)blockIdx.x * kBlock + threadIdx.x;
  v += blockIdx.y * stride;
  if (k >= m) return;
  double a[1 << LV];
#pragma unroll
  for (int i = 0; i < 1 << LV; i++) a[i] = v[k + i * m];
#pragma unroll
  for (int w = 1 << (LV - 1); w > 0; w /= 2)
#pragma unroll
    for (int i = 0; i < w; i++) a[i] += a[i + w];
  v[k] = a[0];
}
// the remaining levels of up to kFoldLast values, in workgroup memory; array
// y's sum to out[y]
constexpr int kFoldLast = 4096;
__global__ __launch_bounds__(1024) void k_fold_last(const double *v, long stride, int n, double *out) {
  __shared__ double s[kFoldLast];
  v += blockIdx.x * stride;
  for (int k = threadIdx.x; k < n; k += 1024) s[k] = v[k];
  __syncthreads();
  while (n > 1) {
    const int j = n / 2, off = n - j;
    for (int k = threadIdx.x; k < j; k += 1024) s[k] += s[k + off];
    __syncthreads();
    n = off;
  }
  if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// The reference's pairwise tree sums of `arrays` arrays of n values (stride
// apart; overwritten) into out[arrays] on the device: two or three launches
// instead of one per level (18 for 2^18 values, 3 us each).
static void pairwise_sums(Context &c, double *v, long n, long stride, int arrays, double *out) {
  while (n > kFoldLast) {
    const int lv = n % 32 == 0 ? 5 : n % 8 == 0 ? 3 : n % 2 == 0 ? 1 : 0;
    const long m = lv ? n >> lv : n / 2;
    const dim3 grid(nblk(m), (unsigned)arrays);
    if (lv == 5) hipLaunchKernelGGL(k_fold_levels<5>, grid, dim3(kBlock), 0, c.stream, v, stride, m);
    else if (lv == 3) hipLaunchKernelGGL(k_fold_levels<3>, grid, dim3(kBlock), 0, c.stream, v, stride, m);
    else if (lv == 1) hipLaunchKernelGGL(k_fold_levels<1>, grid, dim3(kBlock), 0, c.stream, v, stride, m);
    else hipLaunchKernelGGL(k_fold, grid, dim3(kBlock), 0, c.stream, v, stride, m, n - m);
    n = lv ? m : n - m;
  }
  hipLaunchKernelGGL(k_fold_last, dim3((unsigned)arrays), dim3(1024), 0, c.stream, v, stride, (int)n, out);
}

int action_sum(Context &c, double *out) {
  double *sum = (double *)scratch_get(c, SCR_SUMS, sizeof(double));
  if (!sum) return -1;
  pairwise_sums(c, c.action, c.V, c.V, 1, sum);
  return d2h_sync(c, out, sum, sizeof(double)) ? 0 : -1;
}

// ------------------------------------------------------------ measurements
// gaugemeas.cc:6-66 (Conf::calc_plaq): per site minus Re tr of its three
// temporal (nu = 3) and three spatial plaquettes, at the reference site
// index.  A workgroup takes 64 sites, a wave per plane; a tile's four
// workgroups (parity, temporal or spatial) follow each other on one XCD and
// each XCD has a contiguous part of the lattice, so that the links the
// plaquettes share come from its L2.  24^3x6: 17 us (a grid that spread
// neighbouring tiles over the XCDs 28, one thread for all six planes 37).
__global__ __launch_bounds__(192) void k_plaq(LatticeDims L, const double2 *U, double *vt, double *vs) {
  __shared__ double sh[2][64];
  const int lane = threadIdx.x & 63, plane = threadIdx.x >> 6;
  const unsigned b = xcd_block(blockIdx.x, gridDim.x);
  const int spatial = (int)(b & 1u), par = (int)((b >> 1) & 1u);
  const int h = (int)(b >> 2) * 64 + lane;
  const bool in = h < (int)L.Vh;
  // planes (plane, 3), or (0, 1), (0, 2), (1, 2)
  const int mu = __builtin_amdgcn_readfirstlane(spatial ? plane >> 1 : plane);
  const int nu = __builtin_amdgcn_readfirstlane(spatial ? 1 + ((plane + 1) >> 1) : 3);
  const double p = in ? plaq_re(L, U, par, h, site_coords_i(L, par, h), mu, nu) : 0.0;
  if (plane) sh[plane - 1][lane] = p;
  __syncthreads();
  if (plane == 0 && in) (spatial ? vs : vt)[(long)par * L.Vh + h] = -p - sh[0][lane] - sh[1][lane];
}

// gaugemeas.cc:70-104 (Conf::calc_poly): one line per spatial point, from
// the sites r < vol3 (even parity, t = 0 or 1), minus the trace
__global__ __launch_bounds__(kBlock) void k_poly(LatticeDims L, const double2 *U, double *vre, double *vim,
                                                 long vol3) {
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= vol3) return;
  const SiteCoord c = site_coords_i(L, 0, (int)r);
  int t = c.t, par = 0;
  Mat<double> a = load_link_d18(U, L.Vh, 3, 0, r);
  for (int k = 1; k < L.nt; k++) {
    t = t + 1 == L.nt ? 0 : t + 1;
    par ^= 1;
    a = mmul(a, load_link_d18(U, L.Vh, 3, par, half_index_i(L, c.x, c.y, c.z, t)));
  }
  vre[r] = -(a.e[0][0].x + a.e[1][1].x + a.e[2][2].x);
  vim[r] = -(a.e[0][0].y + a.e[1][1].y + a.e[2][2].y);
}

__device__ __forceinline__ uint4 philox4x32(uint4 ctr, uint2 key);

// chiralmeas.cc:18-205 (one noise vector, no imaginary chemical potential)
__global__ __launch_bounds__(kBlock) void k_axpby(double2 *out, const double2 *x, const double2 *y, double a,
                                                  double b, long n) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double2 u = x[i], v = y[i];
  out[i] = make_double2(a * u.x + b * v.x, a * u.y + b * v.y);
}

__global__ __launch_bounds__(kBlock) void k_z2noise(double2 *out, long n, unsigned long long seed,
                                                    unsigned long long stream) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint4 r = philox4x32(make_uint4((unsigned)i, (unsigned)(i >> 32), 7u, (unsigned)stream),
                             make_uint2((unsigned)seed, (unsigned)(seed >> 32)));
  out[i] = make_double2((r.x & 1u) ? -1.0 : 1.0, 0.0);
}

__device__ __forceinline__ double2 cdot3(const double2 *a, long as, const double2 *b, long bs) {
  double2 r = make_double2(0.0, 0.0);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double2 u = a[k * as], v = b[k * bs];
    r.x += u.x * v.x + u.y * v.y;  // conj(u) * v
    r.y += u.x * v.y - u.y * v.x;
  }
  return r;
}
// <w, U v> with U the link at (mu, par, h) and v the spinor at half index hn
__device__ __forceinline__ double2 dot_link(const double2 *w, long ws, const double2 *U, long Vh, int mu, int par,
                                            long h, const double2 *v, long hn) {
  const Mat<double> m = load_link_d18(U, Vh, mu, par, h);
  double2 r = make_double2(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double2 t = make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < 3; k++) cfma(t, m.e[i][k], v[k * Vh + hn]);
    const double2 u = w[i * ws];
    r.x += u.x * t.x + u.y * t.y;
    r.y += u.x * t.y - u.y * t.x;
  }
  return r;
}
// <U w, v> = conj(<v, U w>)
__device__ __forceinline__ double2 dot_link_left(const double2 *U, long Vh, int mu, int par, long h,
                                                 const double2 *w, long hn, const double2 *v, long vs) {
  const double2 r = dot_link(v, vs, U, Vh, mu, par, h, w, hn);
  return make_double2(r.x, -r.y);
}

// per half index i: [chiral re, im, energy re, im, baryon re, im, pressure re, im]
__global__ __launch_bounds__(kBlock) void k_chiral_terms(LatticeDims L, const double2 *U, const double2 *re_,
                                                         const double2 *ro, const double2 *ce, const double2 *co,
                                                         double *w) {
  const long Vh = L.Vh;
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= Vh) return;
  const SiteCoord ce_ = site_coords(L, 0, i), co_ = site_coords(L, 1, i);
  const double2 a = cdot3(ro + i, Vh, co + i, Vh), b = cdot3(re_ + i, Vh, ce + i, Vh);
  double v[8];
  v[0] = a.x + b.x;
  v[1] = a.y + b.y;
  // temporal hops: even i -> odd neighbour, odd i -> even neighbour
  {
    const long ne = neighbour(L, ce_, 3, +1), no = neighbour(L, co_, 3, +1);
    double2 p1 = dot_link(re_ + i, Vh, U, Vh, 3, 0, i, co, ne);
    double2 p2 = dot_link_left(U, Vh, 3, 0, i, ro, ne, ce + i, Vh);
    double2 c1 = make_double2(p1.x - p2.x, p1.y - p2.y), c2 = make_double2(p1.x + p2.x, p1.y + p2.y);
    p1 = dot_link(ro + i, Vh, U, Vh, 3, 1, i, ce, no);
    p2 = dot_link_left(U, Vh, 3, 1, i, re_, no, co + i, Vh);
    c1.x += p1.x - p2.x; c1.y += p1.y - p2.y;
    c2.x += p1.x + p2.x; c2.y += p1.y + p2.y;
    v[2] = c1.x; v[3] = c1.y; v[4] = c2.x; v[5] = c2.y;
  }
  double2 c1 = make_double2(0.0, 0.0);
  for (int k = 0; k < 3; k++) {
    const long ne = neighbour(L, ce_, k, +1), no = neighbour(L, co_, k, +1);
    double2 p = dot_link(re_ + i, Vh, U, Vh, k, 0, i, co, ne);
    c1.x += p.x; c1.y += p.y;
    p = dot_link_left(U, Vh, k, 0, i, ro, ne, ce + i, Vh);
    c1.x -= p.x; c1.y -= p.y;
    p = dot_link(ro + i, Vh, U, Vh, k, 1, i, ce, no);
    c1.x += p.x; c1.y += p.y;
    p = dot_link_left(U, Vh, k, 1, i, re_, no, co + i, Vh);
    c1.x -= p.x; c1.y -= p.y;
  }
  v[6] = c1.x;
  v[7] = c1.y;
#pragma unroll
  for (int k = 0; k < 8; k++) w[k * Vh + i] = v[k];
}

int chiral_meas(Context &c, const double *rnd_e_h, const double *rnd_o_h, unsigned long long seed, double res,
                int max_cg, double n_flavours, double *out, int *iters) {
  const long Vh = c.Vh, n3 = 3 * Vh;
  double2 *buf = (double2 *)scratch_get(c, SCR_MEAS, sizeof(double2) * n3 * 6 + sizeof(double) * (8 * Vh + 8));
  if (!buf) return -1;
  double *w = (double *)(buf + 6 * n3);
  double2 *re_ = buf, *ro = buf + n3, *phi = buf + 2 * n3, *ce = buf + 3 * n3, *co = buf + 4 * n3, *tmp = buf + 5 * n3;
  if (rnd_e_h && rnd_o_h) {
    if (upload_spinors(c, rnd_e_h, re_, 1) || upload_spinors(c, rnd_o_h, ro, 1)) return -1;
  } else {
    hipLaunchKernelGGL(k_z2noise, dim3(nblk(n3)), dim3(kBlock), 0, c.stream, re_, n3, seed, 0ull);
    hipLaunchKernelGGL(k_z2noise, dim3(nblk(n3)), dim3(kBlock), 0, c.stream, ro, n3, seed, 1ull);
  }
  launch_hop_d(c, 0, ro, tmp, 1, n3, n3);  // D_eo rnd_o
  hipLaunchKernelGGL(k_axpby, dim3(nblk(n3)), dim3(kBlock), 0, c.stream, phi, re_, tmp, c.mass, -1.0, n3);
  const double shift0 = 0.0;
  int it = 0;
  const int rc = multishift_solve(c, phi, 1, 1, &shift0, res, 0, PREC_FP64, max_cg, ce, &it);
  if (rc) return rc;
  launch_hop_d(c, 1, ce, tmp, 1, n3, n3);  // D_oe chi_e
  const double im = 1.0 / c.mass;
  hipLaunchKernelGGL(k_axpby, dim3(nblk(n3)), dim3(kBlock), 0, c.stream, co, ro, tmp, im, -im, n3);
  hipLaunchKernelGGL(k_chiral_terms, dim3(nblk(Vh)), dim3(kBlock), 0, c.stream, c.L, c.U64, re_, ro, ce, co, w);
  pairwise_sums(c, w, Vh, Vh, 8, w + 8 * Vh);
  double h[8];
  if (!d2h_sync(c, h, w + 8 * Vh, sizeof(h))) return -1;
  const double inv_size = 1.0 / (double)c.V;
  const double f0 = n_flavours * 0.25 * inv_size, f1 = 0.5 * n_flavours * 0.25 * inv_size;
  out[0] = h[0] * f0; out[1] = h[1] * f0;
  for (int k = 2; k < 8; k++) out[k] = h[k] * f1;
  if (iters) *iters = it;
  return 0;
}

int gauge_meas(Context &c, double *pls, double *plt, double *pre, double *pim) {
  const long vol3 = (long)c.L.nx * c.L.ny * c.L.nz;
  double *w = (double *)scratch_get(c, SCR_MEAS, sizeof(double) * (2 * c.V + 2 * vol3 + 4));
  if (!w) return -1;
  double *vt = w, *vs = w + c.V, *vre = w + 2 * c.V, *vim = vre + vol3, *sums = vim + vol3;
  hipLaunchKernelGGL(k_plaq, dim3((unsigned)((c.Vh + 63) / 64 * 4)), dim3(192), 0, c.stream, c.L, c.U64, vt, vs);
  hipLaunchKernelGGL(k_poly, dim3((unsigned)((vol3 + 63) / 64)), dim3(64), 0, c.stream, c.L, c.U64, vre, vim, vol3);
  pairwise_sums(c, vt, c.V, c.V, 2, sums);
  pairwise_sums(c, vre, vol3, vol3, 2, sums + 2);
  double h[4];
  if (!d2h_sync(c, h, sums, sizeof(h))) return -1;
  // the reference's normalisation order: sum * (1/V/3.) * one_by_three
  const double inv_size_by_three = 1.0 / (double)c.V / 3.;
  const double inv_vol3 = 1.0 / (double)vol3;
  const double one_by_three = 0.3333333333333333333333333333333333333333333333333333333333333333333;
  *plt = h[0] * inv_size_by_three * one_by_three;
  *pls = h[1] * inv_size_by_three * one_by_three;
  *pre = h[2] * inv_vol3 * one_by_three;
  *pim = h[3] * inv_vol3 * one_by_three;
  return 0;
}

// --------------------------------------------------------------------- RNG
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) counter-based generator;
// Box-Muller with radius sqrt(-ln u) gives N(0,1/2) components (gauss.cc:10-35).
__device__ __forceinline__ uint4 philox4x32(uint4 ctr, uint2 key) {
  const unsigned M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; r++) {
    const unsigned long long p0 = (unsigned long long)M0 * ctr.x;
    const unsigned long long p1 = (unsigned long long)M1 * ctr.z;
    const unsigned hi0 = (unsigned)(p0 >> 32), lo0 = (unsigned)p0;
    const unsigned hi1 = (unsigned)(p1 >> 32), lo1 = (unsigned)p1;
    ctr = make_uint4(hi1 ^ ctr.y ^ key.x, lo1, hi0 ^ ctr.w ^ key.y, lo0);
    key.x += W0;
    key.y += W1;
  }
  return ctr;
}
__device__ __forceinline__ double u53(unsigned a, unsigned b) {
  const unsigned long long v = ((unsigned long long)a << 21) ^ (unsigned long long)b;
  return ((double)(v & ((1ull << 53) - 1)) + 0.5) * (1.0 / 9007199254740992.0);
}
__device__ __forceinline__ double2 gauss_pair(unsigned long long seed, unsigned long long stream, unsigned long long idx,
                                              unsigned k) {
  const uint4 r = philox4x32(make_uint4((unsigned)idx, (unsigned)(idx >> 32), k, (unsigned)stream),
                             make_uint2((unsigned)seed, (unsigned)(seed >> 32)));
  const double u1 = u53(r.x, r.y), u2 = u53(r.z, r.w);
  const double rad = sqrt(-log(u1));
  double sn, cs;
  sincos(6.283185307179586476925286766559 * u2, &sn, &cs);
  return make_double2(rad * cs, rad * sn);
}

// gauss.cc:63-86 layout of the gaussian su(3) matrix
__global__ __launch_bounds__(kBlock) void k_gauss_mom(double2 *P, long Vh, unsigned long long seed,
                                                      unsigned long long stream) {
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int par = blockIdx.y, mu = blockIdx.z;
  if (h >= Vh) return;
  const unsigned long long link = ((unsigned long long)mu * 2 + par) * (unsigned long long)Vh + h;
  double r[8];
  for (int k = 0; k < 4; k++) {
    const double2 g = gauss_pair(seed, stream, link, k);
    r[2 * k] = g.x;
    r[2 * k + 1] = g.y;
  }
  const double s3 = 0.57735026918962576450914878050196;
  double2 *b = P + (long)(mu * 2 + par) * 4 * Vh + h;
  b[0] = make_double2(r[0], -r[1]);
  b[Vh] = make_double2(r[3], -r[4]);
  b[2 * Vh] = make_double2(r[5], -r[6]);
  b[3 * Vh] = make_double2(r[2] + s3 * r[7], -r[2] + s3 * r[7]);
}

int gauss_momenta(Context &c, unsigned long long seed, unsigned long long stream) {
  hipLaunchKernelGGL(k_gauss_mom, dim3(nblk(c.Vh), 2, 4), dim3(kBlock), 0, c.stream, c.P, c.Vh, seed, stream);
  return hip_ok(c, hipGetLastError(), "gauss momenta") ? 0 : -1;
}

__global__ __launch_bounds__(kBlock) void k_gauss_spinor(double2 *out, long Vh, unsigned long long seed,
                                                         unsigned long long stream) {
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int ps = blockIdx.y;
  if (h >= Vh) return;
  for (int k = 0; k < 3; k++)
    out[((long)ps * 3 + k) * Vh + h] = gauss_pair(seed, stream, (unsigned long long)ps * Vh + h, k);
}

int gauss_spinor(Context &c, double2 *out, int n, unsigned long long seed, unsigned long long stream) {
  hipLaunchKernelGGL(k_gauss_spinor, dim3(nblk(c.Vh), n), dim3(kBlock), 0, c.stream, out, c.Vh, seed, stream);
  return hip_ok(c, hipGetLastError(), "gauss spinor") ? 0 : -1;
}

// ------------------------------------------------ reversibility distances
// revupdate.cc:66-92: sum over links of l2norm2(U - U_save) (kind 0: FP64
// 18-real links, n = 72 Vh complex entries) or of l2norm2(P + P_save) (kind
// 1: hermitian algebra fields stored as P01, P02, P12, (P00, P11), n = 32 Vh;
// the full 3x3 norm counts each off-diagonal entry twice and P22 = -(P00 +
// P11)).  One FP64 partial per workgroup, summed in a fixed order by one
// workgroup.
__global__ __launch_bounds__(kBlock) void k_pair_norm2(const double2 *a, const double2 *b, long Vh, int kind,
                                                       double *partial) {
  __shared__ double sh[kBlock / 64];
  const long stride = (long)gridDim.x * kBlock;
  double v = 0.0;
  if (kind == 0) {
    const long n = 72 * Vh;
    for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
      const double2 x = a[i], y = b[i];
      const double dx = x.x - y.x, dy = x.y - y.y;
      v += dx * dx + dy * dy;
    }
  } else {
    const long n = 8 * Vh;  // (mu, parity, h)
    for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
      const long blk = i / Vh, h = i - blk * Vh;
      double2 d[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const double2 x = a[(blk * 4 + k) * Vh + h], y = b[(blk * 4 + k) * Vh + h];
        d[k] = make_double2(x.x + y.x, x.y + y.y);
      }
      const double p22 = d[3].x + d[3].y;
      v += 2.0 * (d[0].x * d[0].x + d[0].y * d[0].y + d[1].x * d[1].x + d[1].y * d[1].y + d[2].x * d[2].x +
                  d[2].y * d[2].y) +
           d[3].x * d[3].x + d[3].y * d[3].y + p22 * p22;
    }
  }
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int k = 0; k < kBlock / 64; k++) s += sh[k];
    partial[blockIdx.x] = s;
  }
}

__global__ __launch_bounds__(kBlock) void k_sum_partials(const double *partial, int n, double *out) {
  __shared__ double sh[kBlock / 64];
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += kBlock) v += partial[i];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int k = 0; k < kBlock / 64; k++) s += sh[k];
    *out = s;
  }
}

int pair_norm2(Context &c, const double2 *a, const double2 *b, int kind, double *out) {
  const int nb = 1024;
  double *part = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&part, sizeof(double) * (nb + 1), c.stream), "pair norm")) return -1;
  hipLaunchKernelGGL(k_pair_norm2, dim3(nb), dim3(kBlock), 0, c.stream, a, b, c.Vh, kind, part);
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kBlock), 0, c.stream, part, nb, part + nb);
  hipMemcpyAsync(out, part + nb, sizeof(double), hipMemcpyDeviceToHost, c.stream);
  hipFreeAsync(part, c.stream);
  return hip_ok(c, hipStreamSynchronize(c.stream), "pair norm") ? 0 : -1;
}

// ------------------------------------------------------- copy probe
// plain streaming copy of known size: calibrates the HBM byte counters and
// gives the achievable-bandwidth reference for the roofline
__global__ __launch_bounds__(kBlock) void k_copy_probe(const double4 *__restrict__ in, double4 *__restrict__ out,
                                                       long n) {
  const long stride = (long)gridDim.x * kBlock;
  for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) out[i] = in[i];
}

int time_copy(Context &c, size_t bytes, int reps, double *ms) {
  const long n = (long)(bytes / sizeof(double4));
  double4 *a = nullptr, *b = nullptr;
  if (!hip_ok(c, hipMalloc(&a, n * sizeof(double4)), "copy probe")) return -1;
  if (!hip_ok(c, hipMalloc(&b, n * sizeof(double4)), "copy probe")) { hipFree(a); return -1; }
  hipMemsetAsync(a, 0, n * sizeof(double4), c.stream);
  const unsigned nb = 256 * 8 * 4;
  hipLaunchKernelGGL(k_copy_probe, dim3(nb), dim3(kBlock), 0, c.stream, a, b, n);
  hipEvent_t e0, e1;
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  hipEventRecord(e0, c.stream);
  for (int r = 0; r < reps; r++)
    hipLaunchKernelGGL(k_copy_probe, dim3(nb), dim3(kBlock), 0, c.stream, (r & 1) ? b : a, (r & 1) ? a : b, n);
  hipEventRecord(e1, c.stream);
  hipEventSynchronize(e1);
  float t = 0.f;
  hipEventElapsedTime(&t, e0, e1);
  *ms = (double)t / reps;
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  hipFree(a);
  hipFree(b);
  return hip_ok(c, hipGetLastError(), "copy probe") ? 0 : -1;
}

// ----------------------------------------------------- host-layout transfers
// Large copies between the caller's (pageable) arrays and device memory.  The
// runtime's own pageable copy is one thread that copies through its pinned
// buffers and takes the page faults of a fresh destination: 151 MB (the
// links or momenta of 32^3x8) to the host took 15 ms, 9 ms into pages that
// exist, 5.4 ms to the device.  Here kStageThreads threads take chunks in
// turn, each with two pinned buffers (the copy of one chunk over the bus
// while the other is moved by the CPU): 4.4 ms and 4.0 ms; the bus alone
// takes 2.8 ms, and more threads or larger chunks gain nothing.
//
// The pinned buffers (16 MB) serve every context of a device, one transfer
// at a time (the bus is theirs), and are freed with the last of them.
// Allocating them takes 3.5 ms, as long as they save on some 50 MB, so they
// are allocated by the transfer that brings the large ones' total past
// kStageWorth.  Memory that the runtime knows (pinned or managed) takes its
// own copy, which goes over the bus directly.
constexpr int kStageThreads = 4;
constexpr size_t kStageChunk = 2u << 20;
constexpr size_t kStageMin = 8u << 20;  // smaller copies: the runtime's (two chunks a thread and more)
constexpr size_t kStageWorth = 64u << 20;

struct HostStage {
  std::mutex m;  // buf and moved; held through a transfer
  char *buf = nullptr;
  size_t moved = 0;  // bytes of the large transfers
  std::atomic<int> users{0};
};
static HostStage &host_stage(int device) {
  static HostStage s[64];
  return s[device < 0 || device >= 64 ? 0 : device];
}
void host_stage_retain(int device) { host_stage(device).users++; }
void host_stage_release(int device) {
  HostStage &s = host_stage(device);
  if (--s.users) return;
  std::lock_guard<std::mutex> l(s.m);
  if (s.users) return;  // a context made meanwhile
  if (s.buf) hipHostFree(s.buf);
  s.buf = nullptr;
  s.moved = 0;
}

static bool known_to_runtime(const void *p) {
  hipPointerAttribute_t a = {};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// whether a copy goes through the pinned buffers, which are there then (the
// context, a user of them, keeps them)
static bool host_staged(HostStage &s, const void *host, size_t bytes) {
  if (bytes < kStageMin || known_to_runtime(host)) return false;
  std::lock_guard<std::mutex> l(s.m);
  if (s.moved <= kStageWorth) s.moved += bytes;
  if (!s.buf && s.moved > kStageWorth &&
      hipHostMalloc((void **)&s.buf, 2 * kStageThreads * kStageChunk, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    s.buf = nullptr;
  }
  return s.buf != nullptr;
}

// dev -> host (down) or host -> dev on c.stream; every caller synchronises
// the stream before it returns to the user
static bool host_copy(Context &c, void *dev, void *host, size_t bytes, bool down) {
  HostStage &s = host_stage(c.device);
  if (!host_staged(s, host, bytes)) {
    const hipError_t e = down ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, c.stream)
                              : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, c.stream);
    return hip_ok(c, e, "host transfer");
  }
  // the stream's earlier work is over before the buffers are taken: others
  // wait for a transfer, not for what it follows
  if (!hip_ok(c, hipStreamSynchronize(c.stream), "host transfer")) return false;
  std::lock_guard<std::mutex> l(s.m);
  c.path[RHMC_COUNT_STAGED]++;
  const size_t n = (bytes + kStageChunk - 1) / kStageChunk;
  std::atomic<size_t> next{0};
  std::atomic<bool> ok{true};
  auto size = [&](size_t i) { return std::min(kStageChunk, bytes - i * kStageChunk); };
  auto worker = [&](int k) {
    hipEvent_t ev[2] = {};
    bool good = hipSetDevice(c.device) == hipSuccess;
    for (auto &e : ev) good = good && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    char *b[2] = {s.buf + (size_t)(2 * k) * kStageChunk, s.buf + (size_t)(2 * k + 1) * kStageChunk};
    size_t at[2] = {n, n};
    if (down) {
      auto issue = [&](int q) {
        at[q] = next++;
        if (!good || at[q] >= n) return;
        good = hipMemcpyAsync(b[q], (char *)dev + at[q] * kStageChunk, size(at[q]), hipMemcpyDeviceToHost, c.stream) ==
                   hipSuccess &&
               hipEventRecord(ev[q], c.stream) == hipSuccess;
      };
      issue(0);
      issue(1);
      for (int q = 0; good && at[q] < n; q ^= 1) {
        good = hipEventSynchronize(ev[q]) == hipSuccess;
        if (good) memcpy((char *)host + at[q] * kStageChunk, b[q], size(at[q]));
        issue(q);
      }
    } else {
      for (int q = 0; good; q ^= 1) {
        const bool used = at[q] < n;
        const size_t i = next++;
        if (i >= n) break;
        if (used) good = hipEventSynchronize(ev[q]) == hipSuccess;
        at[q] = i;
        if (!good) break;
        memcpy(b[q], (const char *)host + i * kStageChunk, size(i));
        good = hipMemcpyAsync((char *)dev + i * kStageChunk, b[q], size(i), hipMemcpyHostToDevice, c.stream) ==
                   hipSuccess &&
               hipEventRecord(ev[q], c.stream) == hipSuccess;
      }
    }
    // nothing of this worker's buffers in flight when it ends
    for (int q = 0; q < 2; q++) {
      if (ev[q] && at[q] < n) good = hipEventSynchronize(ev[q]) == hipSuccess && good;
      if (ev[q]) hipEventDestroy(ev[q]);
    }
    if (!good) ok = false;
  };
  // the calling thread works too, so a thread that cannot be started only
  // leaves its chunks to the others
  std::thread th[kStageThreads - 1];
  try {
    for (int k = 1; k < kStageThreads; k++) th[k - 1] = std::thread(worker, k);
  } catch (const std::exception &) {
  }
  worker(0);
  for (std::thread &t : th)
    if (t.joinable()) t.join();
  if (!ok) {
    (void)hipStreamSynchronize(c.stream);
    c.last_error = "host transfer failed";
  }
  return ok;
}

// host links/algebra: [4V][3][3] complex at mu*V + par*Vh + h  ==  [(mu*2+par)*Vh + h]
__global__ __launch_bounds__(kBlock) void k_links_in(const double2 *aos, double2 *U, long Vh) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;  // over 8*Vh links
  if (i >= 8 * Vh) return;
  const long blk = i / Vh, h = i - blk * Vh;
#pragma unroll
  for (int k = 0; k < 9; k++) U[(blk * 9 + k) * Vh + h] = aos[i * 9 + k];
}
__global__ __launch_bounds__(kBlock) void k_links_out(const double2 *U, double2 *aos, long Vh) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= 8 * Vh) return;
  const long blk = i / Vh, h = i - blk * Vh;
#pragma unroll
  for (int k = 0; k < 9; k++) aos[i * 9 + k] = U[(blk * 9 + k) * Vh + h];
}
// algebra fields: full matrix -> 8-real packing (herm: real diag, aherm: imag diag)
__global__ __launch_bounds__(kBlock) void k_alg_in(const double2 *aos, double2 *A, long Vh, int herm) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= 8 * Vh) return;
  const long blk = i / Vh, h = i - blk * Vh;
  const double2 *m = aos + i * 9;
  double2 *b = A + blk * 4 * Vh + h;
  b[0] = m[1];
  b[Vh] = m[2];
  b[2 * Vh] = m[5];
  b[3 * Vh] = herm ? make_double2(m[0].x, m[4].x) : make_double2(m[0].y, m[4].y);
}
__global__ __launch_bounds__(kBlock) void k_alg_out(const double2 *A, double2 *aos, long Vh, int herm) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= 8 * Vh) return;
  const long blk = i / Vh, h = i - blk * Vh;
  const int mu = (int)(blk / 2), par = (int)(blk % 2);
  const Mat<double> m = herm ? load_herm(A, Vh, mu, par, h) : load_aherm(A, Vh, mu, par, h);
  double2 *o = aos + i * 9;
  for (int r = 0; r < 3; r++)
    for (int k = 0; k < 3; k++) o[r * 3 + k] = m.e[r][k];
}
// spinors: host [n][Vh][3] <-> device [n][3][Vh]
__global__ __launch_bounds__(kBlock) void k_spin_in(const double2 *aos, double2 *v, long Vh) {
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int j = blockIdx.y;
  if (h >= Vh) return;
  for (int k = 0; k < 3; k++) v[((long)j * 3 + k) * Vh + h] = aos[((long)j * Vh + h) * 3 + k];
}
__global__ __launch_bounds__(kBlock) void k_spin_out(const double2 *v, double2 *aos, long Vh) {
  const long h = (long)blockIdx.x * kBlock + threadIdx.x;
  const int j = blockIdx.y;
  if (h >= Vh) return;
  for (int k = 0; k < 3; k++) aos[((long)j * Vh + h) * 3 + k] = v[((long)j * 3 + k) * Vh + h];
}

// Largest |row 2 - eta (row 0 x row 1)^*| over the links, per workgroup, on
// the host layout (link i = (2 mu + parity) Vh + h).  The 12-real copies
// (the FP32 MD operator, the FP64 solves, the gauge force) rebuild row 2
// this way, which reproduces the stored link only when it is unitary.  NaN
// entries are skipped (the solvers report them).
__global__ __launch_bounds__(kBlock) void k_unitarity(LatticeDims L, const double2 *aos, double *part) {
  __shared__ double red[kBlock];
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  double d = 0.0;
  if (i < 8 * L.Vh) {
    const long blk = i / L.Vh, h = i - blk * L.Vh;
    const int mu = (int)(blk / 2), par = (int)(blk % 2);
    Mat<double> m;
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k / 3][k % 3] = aos[i * 9 + k];
    const SiteCoord c = site_coords_i(L, par, (int)h);
    Mat<double> r = m;
    rebuild_row2(r, (double)eta_phase(L, c.x, c.y, c.z, c.t, mu));
#pragma unroll
    for (int k = 0; k < 3; k++) d = fmax(d, hypot(r.e[2][k].x - m.e[2][k].x, r.e[2][k].y - m.e[2][k].y));
  }
  red[threadIdx.x] = d;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Links from the host layout to dst (FP64 18-real).  *max_dev receives the
// largest deviation from unitarity (k_unitarity); above tol dst is left
// unchanged and 1 is returned.
int upload_links(Context &c, const double *host, double2 *dst, double tol, double *max_dev) {
  const size_t bytes = sizeof(double2) * 9 * 8 * c.Vh;
  const unsigned nb = nblk(8 * c.Vh);
  double2 *st = nullptr;
  double *part = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  if (!hip_ok(c, hipMallocAsync((void **)&part, sizeof(double) * nb, c.stream), "stage")) {
    hipFreeAsync(st, c.stream);
    return -1;
  }
  const bool copied = host_copy(c, st, const_cast<double *>(host), bytes, false);
  hipLaunchKernelGGL(k_unitarity, dim3(nb), dim3(kBlock), 0, c.stream, c.L, st, part);
  std::vector<double> hp(nb);
  hipMemcpyAsync(hp.data(), part, sizeof(double) * nb, hipMemcpyDeviceToHost, c.stream);
  hipFreeAsync(part, c.stream);
  if (!hip_ok(c, hipStreamSynchronize(c.stream), "upload links") || !copied) {
    hipFreeAsync(st, c.stream);
    return -1;
  }
  double m = 0.0;
  for (double v : hp) m = std::max(m, v);
  *max_dev = m;
  if (m > tol) {
    hipFreeAsync(st, c.stream);
    return hip_ok(c, hipStreamSynchronize(c.stream), "upload links") ? 1 : -1;
  }
  hipLaunchKernelGGL(k_links_in, dim3(nblk(8 * c.Vh)), dim3(kBlock), 0, c.stream, st, dst, c.Vh);
  hipFreeAsync(st, c.stream);
  return hip_ok(c, hipStreamSynchronize(c.stream), "upload links") ? 0 : -1;
}
int download_links(Context &c, const double2 *src, double *host) {
  const size_t bytes = sizeof(double2) * 9 * 8 * c.Vh;
  double2 *st = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  hipLaunchKernelGGL(k_links_out, dim3(nblk(8 * c.Vh)), dim3(kBlock), 0, c.stream, src, st, c.Vh);
  const bool copied = host_copy(c, st, host, bytes, true);
  hipFreeAsync(st, c.stream);
  return copied && hip_ok(c, hipStreamSynchronize(c.stream), "download links") ? 0 : -1;
}
int upload_alg(Context &c, const double *host, double2 *dst, int herm) {
  const size_t bytes = sizeof(double2) * 9 * 8 * c.Vh;
  double2 *st = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  const bool copied = host_copy(c, st, const_cast<double *>(host), bytes, false);
  hipLaunchKernelGGL(k_alg_in, dim3(nblk(8 * c.Vh)), dim3(kBlock), 0, c.stream, st, dst, c.Vh, herm);
  hipFreeAsync(st, c.stream);
  return copied && hip_ok(c, hipStreamSynchronize(c.stream), "upload algebra") ? 0 : -1;
}
int download_alg(Context &c, const double2 *src, double *host, int herm) {
  const size_t bytes = sizeof(double2) * 9 * 8 * c.Vh;
  double2 *st = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  hipLaunchKernelGGL(k_alg_out, dim3(nblk(8 * c.Vh)), dim3(kBlock), 0, c.stream, src, st, c.Vh, herm);
  const bool copied = host_copy(c, st, host, bytes, true);
  hipFreeAsync(st, c.stream);
  return copied && hip_ok(c, hipStreamSynchronize(c.stream), "download algebra") ? 0 : -1;
}
int upload_spinors(Context &c, const double *host, double2 *dst, int n) {
  const size_t bytes = sizeof(double2) * 3 * c.Vh * n;
  double2 *st = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  const bool copied = host_copy(c, st, const_cast<double *>(host), bytes, false);
  hipLaunchKernelGGL(k_spin_in, dim3(nblk(c.Vh), n), dim3(kBlock), 0, c.stream, st, dst, c.Vh);
  hipFreeAsync(st, c.stream);
  return copied && hip_ok(c, hipStreamSynchronize(c.stream), "upload spinors") ? 0 : -1;
}
int download_spinors(Context &c, const double2 *src, double *host, int n) {
  const size_t bytes = sizeof(double2) * 3 * c.Vh * n;
  double2 *st = nullptr;
  if (!hip_ok(c, hipMallocAsync((void **)&st, bytes, c.stream), "stage")) return -1;
  hipLaunchKernelGGL(k_spin_out, dim3(nblk(c.Vh), n), dim3(kBlock), 0, c.stream, src, st, c.Vh);
  const bool copied = host_copy(c, st, host, bytes, true);
  hipFreeAsync(st, c.stream);
  return copied && hip_ok(c, hipStreamSynchronize(c.stream), "download spinors") ? 0 : -1;
}

}  // namespace rhmc
