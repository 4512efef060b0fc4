// resident.hpp -- the stored-basis multi-shift CG of small lattices as one
// launch (included by solver.hip).
//
// On a lattice of a few thousand to ~3 10^4 half sites the two launches of a
// CG iteration are bound by latency: each waits for the launch before it to
// drain, starts its workgroups, fetches its operands and reduces.  Here the
// whole iteration loop runs in one grid whose workgroups are all resident:
// four lanes per site (lane mu its direction, as in k_dslash_ls), P sites of
// each parity per lane, the links of the next half step loaded while the
// sums of this one travel.
//
// Between the two half steps of an iteration the grid meets in an
// all-to-all reduction (res_arrive / res_wait): every workgroup stores its
// partial sum into its own slot and each workgroup reads all slots, adding
// them in one fixed order.  A slot that still holds the sentinel has not
// arrived, so the exchange of the sums is the barrier.  Each XCD reads its
// own copy of the slots, 16 to a line and the lines 256 bytes apart: one
// copy polled by 256 workgroups took 4.2-4.8 us per meeting, eight 2.9-3.0
// (16 workgroups: 1.6 and 1.4).
//
// Visibility between workgroups without cache write-backs or invalidations:
// * spinors are stored with agent-scope atomic stores, which write through
//   the XCD's L2, and the wave waits for them (vmcnt 0) before its workgroup
//   stores its partial;
// * they are read with ordinary loads, from addresses that nothing has read
//   since the launch began: r^(k) is a new basis slot and h of iteration k
//   has a slot of its own, both multiples of the 128-byte cache line, so
//   no L1 or L2 can hold an older copy of a line;
// * partials and the abort flag are read with agent-scope atomic loads.
//
// A wait is bounded (ResGroup::wait; 0: up at the first empty slot): when it
// runs out (the grid is not
// resident because another process holds the device) the workgroup sets the
// abort flag and leaves, the others follow, and the host repeats the solve
// with the per-iteration launches.
#pragma once

#include "resident_plan.hpp"

namespace rhmc {

constexpr int kResAborted = 2;            // MsState::nonfinite of system 0: the grid gave up
constexpr int kResRing = 4;               // reduction slots in use in turn
constexpr int kResCopies = 8;             // copies of the slots, one per XCD
constexpr unsigned long long kResNone = ~0ull;  // a partial that has not arrived
// Bound of a wait: 50 ms of the 100 MHz wall clock.  A meeting takes 1.4-3 us
// and a whole solve a few milliseconds: a workgroup that has not come by then
// has no place on the device.
constexpr long long kResWaitTicks = 5000000ll;
constexpr int kResMaxWaves = 8;           // waves of a workgroup (512 lanes)

// one member of a launch: nvec right-hand sides of one lattice's solve
struct ResArgs {
  LatticeDims L;
  const void *U;
  void *basis, *h;       // slots of stride elements: r^(k) at slot k, h of iteration k at slot k-1
  long stride;           // right-hand sides of the whole solve * 3 * Vh
  const double *diag;    // per system m^2 + its shift
  const BmsShared *sh;   // rho_0 and the zero-source stops of the set-up
  MsState *ms;
  BmsHist *hist;
  unsigned long long *part;  // [kResRing][nvec][kResCopies][copy], res_copy(nwg) each
  int *abort;
  int nvec, nshift, cap, nwg;
  int sites;             // sites of each parity per lane (1 or 2)
};

// one copy of the slots of nwg workgroups: 16 per 128-byte line, a line per 256 bytes
__host__ __device__ __forceinline__ int res_copy(int nwg) { return (nwg + 15) / 16 * 32; }
__device__ __forceinline__ int res_slot(int wg) { return (wg >> 4) * 32 + (wg & 15); }

__device__ __forceinline__ unsigned long long res_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_store(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_put(float2 *p, float2 v) {
  res_store((unsigned long long *)p,
            ((unsigned long long)__float_as_uint(v.y) << 32) | (unsigned long long)__float_as_uint(v.x));
}
__device__ __forceinline__ void res_put(double2 *p, double2 v) {
  res_store((unsigned long long *)p, (unsigned long long)__double_as_longlong(v.x));
  res_store((unsigned long long *)p + 1, (unsigned long long)__double_as_longlong(v.y));
}

template <int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_double(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// wave sum in register moves (quads, 8, 16 lanes by DPP, then the four rows
// read as scalars): the shuffles of wave_sum go through LDS, six in a row
__device__ __forceinline__ double wave_sum_dpp(double v) {
  v += dpp_double<0xB1>(v);   // lanes 1,0,3,2 of each quad
  v += dpp_double<0x4E>(v);   // lanes 2,3,0,1
  v += dpp_double<0x141>(v);  // mirrored half row
  v += dpp_double<0x140>(v);  // mirrored row
  return (lane_double(v, 0) + lane_double(v, 16)) + (lane_double(v, 32) + lane_double(v, 48));
}

// the workgroup's scalars: sums, the base CG's and, one shift per lane, the
// shifted recurrences (bms_step's, carried here instead of in MsState)
template <int NR>
struct ResShared {
  double wave[2][kResMaxWaves][NR];  // wave sums: own partial, all partials
  double diag[NR], rho1[NR], rho2[NR], beta[NR], alpha[NR];
  double coef[2][NR];                // alpha and c of the residual update
  int stop[NR], next[NR];            // stopped before this / the next iteration
  int aborted;
  double z1[NR][kMaxShifts], z2[NR][kMaxShifts], shift[NR][kMaxShifts];
  int flag[NR][kMaxShifts], its[NR][kMaxShifts];
  double omega[NR], omega_prev[NR], gammag[NR], delta[NR], res[NR];
  int iter[NR], nact[NR], bad[NR], max_iter[NR];
};

// stores the workgroup's partial sums of phase p, its spinor stores complete
template <int NR>
__device__ __forceinline__ void res_arrive(const ResArgs &a, ResShared<NR> &s, int wg, int p, const double (&v)[NR]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const double q = wave_sum_dpp(v[r]);
    if (lane == 0) s.wave[0][w][r] = q;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  const int r = threadIdx.x / kResCopies;
  if (r < a.nvec) {
    double q = 0.0;
    for (int k = 0; k < nw; k++) q += s.wave[0][k][r];
    unsigned long long b = (unsigned long long)__double_as_longlong(q);
    if (b == kResNone) b = 0x7ff8000000000000ull;  // a NaN, but not the sentinel
    res_store(a.part + ((long)(p % kResRing) * a.nvec * kResCopies + threadIdx.x) * res_copy(a.nwg) + res_slot(wg), b);
  }
}

// all workgroups' sums of phase p into s.wave[1] (to be added over the
// waves); false when the grid gave up.  Ends with a workgroup barrier.
template <int NR>
__device__ __forceinline__ bool res_wait(const ResArgs &a, ResShared<NR> &s, int wg, int copy, long long wait,
                                         int p) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long cs = res_copy(a.nwg);
  const unsigned long long *row = a.part + ((long)(p % kResRing) * a.nvec * kResCopies + copy) * cs;
  double v[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) v[r] = 0.0;
  for (int i = threadIdx.x; i < a.nwg; i += blockDim.x) {
    const unsigned long long *q = row + res_slot(i);
    unsigned long long b[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) b[r] = r < a.nvec ? res_load(q + r * kResCopies * cs) : 0ull;
    long long t0 = 0;
    for (int n = 0;; n++) {
      bool none = false;
#pragma unroll
      for (int r = 0; r < NR; r++) none |= b[r] == kResNone;
      if (!none) break;
      if (n == 0) t0 = wall_clock64();
      if (((n & 63) == 63 || wait == 0) &&
          (wall_clock64() - t0 >= wait ||
           __hip_atomic_load(a.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        __hip_atomic_store(a.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s.aborted = 1;
        break;
      }
#pragma unroll
      for (int r = 0; r < NR; r++)
        if (b[r] == kResNone) b[r] = res_load(q + r * kResCopies * cs);
    }
#pragma unroll
    for (int r = 0; r < NR; r++) v[r] += __longlong_as_double((long long)b[r]);
  }
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const double q = wave_sum_dpp(v[r]);
    if (lane == 0) s.wave[1][w][r] = q;
  }
  __syncthreads();
  // every workgroup has arrived at p, so all have read phase p-1: its slots
  // are cleared here, three phases before their next use and complete
  // (vmcnt 0) before this workgroup's next arrival
  if (p > 0 && (int)threadIdx.x / kResCopies < a.nvec)
    res_store(a.part + ((long)((p - 1) % kResRing) * a.nvec * kResCopies + threadIdx.x) * cs + res_slot(wg), kResNone);
  return !s.aborted;
}

// sentinel into every slot, before the launch
__global__ __launch_bounds__(kBlock) void k_res_init(unsigned long long *part, int n, int *abort) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) part[i] = kResNone;
  if (blockIdx.x == 0 && threadIdx.x == 0) *abort = 0;
}

// a lane's hop at one site: byte offsets of the neighbours' spinors and of
// the two links (32 bits: the link array of these lattices is below 4 GB),
// the links' phases
template <typename R>
struct ResHop {
  unsigned fo, bo, fl, bl;
  R ef, eb;
};
template <typename R, int LINK>
struct ResLinks {
  LinkRaw<R, LINK> fw, bw;
};

template <typename R, int LINK>
__device__ __forceinline__ void res_hop_setup(const ResArgs &a, int par, int h, int mu, ResHop<R> &o) {
  using T = typename LinkRaw<R, LINK>::T;
  constexpr int N = LinkRaw<R, LINK>::N;
  const SiteCoord c = site_coords_i(a.L, par, h);
  const int hf = neighbour_i(a.L, c, mu, +1), hb = neighbour_i(a.L, c, mu, -1);
  const unsigned Vh = (unsigned)a.L.Vh;
  o.fo = (unsigned)hf * (unsigned)sizeof(Cx<R>);
  o.bo = (unsigned)hb * (unsigned)sizeof(Cx<R>);
  o.fl = ((unsigned)(mu * 2 + par) * N * Vh + (unsigned)h) * (unsigned)sizeof(T);
  o.bl = ((unsigned)(mu * 2 + 1 - par) * N * Vh + (unsigned)hb) * (unsigned)sizeof(T);
  o.ef = (R)eta_phase(a.L, c.x, c.y, c.z, c.t, mu);
  const int tm = (mu == 3) ? (c.t == 0 ? a.L.nt - 1 : c.t - 1) : c.t;
  o.eb = (R)eta_phase(a.L, c.x, c.y, c.z, tm, mu);
}

template <typename R, int LINK>
__device__ __forceinline__ void res_links(const ResArgs &a, const ResHop<R> &o, ResLinks<R, LINK> &l) {
  using T = typename LinkRaw<R, LINK>::T;
  constexpr int N = LinkRaw<R, LINK>::N;
#pragma unroll
  for (int k = 0; k < N; k++) {
    l.fw.e[k] = ld_off((const T *)a.U + (long)k * a.L.Vh, o.fl);
    l.bw.e[k] = ld_off((const T *)a.U + (long)k * a.L.Vh, o.bl);
  }
}

// keeps held links as the 12 reals they were loaded as: without it the row-2
// rebuild, the same in every iteration, is moved out of the loop and its
// results held too (50% more registers)
template <typename R, int LINK>
__device__ __forceinline__ void res_keep(ResLinks<R, LINK> &l) {
#pragma unroll
  for (int k = 0; k < LinkRaw<R, LINK>::N; k++) {
    asm volatile("" : "+v"(l.fw.e[k].x), "+v"(l.fw.e[k].y), "+v"(l.bw.e[k].x), "+v"(l.bw.e[k].y));
    if constexpr (LINK == LINK_S12)
      asm volatile("" : "+v"(l.fw.e[k].z), "+v"(l.fw.e[k].w), "+v"(l.bw.e[k].z), "+v"(l.bw.e[k].w));
  }
}

// the site's hop for NB right-hand sides from r0 on, summed over the quad:
// lane mu < 3 returns colour mu
template <typename R, int LINK, int NB>
__device__ __forceinline__ void res_hop(const ResHop<R> &o, const ResLinks<R, LINK> &l, const Cx<R> *in, long Vh,
                                        int r0, int nvec, int mu, Cx<R> (&out)[NB]) {
  Cx<R> vf[NB][3], vb[NB][3];
#pragma unroll
  for (int q = 0; q < NB; q++) {
    const Cx<R> *v = in + (long)(r0 + q < nvec ? r0 + q : nvec - 1) * 3 * Vh;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      vf[q][i] = ld_off(v + (long)i * Vh, o.fo);
      vb[q][i] = ld_off(v + (long)i * Vh, o.bo);
    }
  }
  const Mat<R> F = link_raw_mat<R, LINK>(l.fw, o.ef), B = link_raw_mat<R, LINK>(l.bw, o.eb);
#pragma unroll
  for (int q = 0; q < NB; q++) {
    Cx<R> acc[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      acc[i] = mk<R>(0, 0);
      cfma(acc[i], F.e[i][0], vf[q][0]);
      cfma(acc[i], F.e[i][1], vf[q][1]);
      cfma(acc[i], F.e[i][2], vf[q][2]);
      cfmsc(acc[i], B.e[0][i], vb[q][0]);
      cfmsc(acc[i], B.e[1][i], vb[q][1]);
      cfmsc(acc[i], B.e[2][i], vb[q][2]);
      acc[i].x = quad_sum(acc[i].x);
      acc[i].y = quad_sum(acc[i].y);
    }
    out[q] = pick3(acc[0], acc[1], acc[2], mu);
  }
}

// workgroup wg of a.nwg: all iterations of one lattice's solve; copy: the
// slots this workgroup reads
template <typename R, int LINK, int NR, int P>
__device__ __forceinline__ void res_body(const ResArgs &a, int wg, int copy, long long wait) {
  using C = Cx<R>;
  // right-hand sides whose operands are in flight together
  constexpr int NB = sizeof(R) == 4 ? (NR < 4 ? NR : 4) : (NR < 2 ? NR : 2);
  // one site per lane: its four links stay in registers for the whole solve
  // (kHeld: FP64 with one system, FP32), else the two of the next half step are
  // loaded while the sums travel (kAhead); two sites load them at the hop
  constexpr bool kHeld = P == 1 && (sizeof(R) == 4 ? NR <= 4 : NR == 1);
  constexpr bool kAhead = P == 1 && !kHeld;
  __shared__ ResShared<NR> s;
  const long Vh = a.L.Vh;
  const int mu = threadIdx.x & 3, lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int spw = blockDim.x >> 2;
  bool mine[P];
  unsigned own[P];  // element of this lane's colour within a vector
  ResHop<R> odd[P], even[P];
  R dg[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) dg[r] = (R)a.diag[r < a.nvec ? r : a.nvec - 1];
  C rv[P][NR], qv[P][NR];  // this lane's colour of r^(k-1) and r^(k-2)
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int site = (wg * P + p) * spw + (int)(threadIdx.x >> 2);
    const bool valid = site < (int)Vh;
    const int h = valid ? site : (int)Vh - 1;
    mine[p] = valid && mu < 3;
    own[p] = (unsigned)((mu < 3 ? mu : 2) * Vh + h);
    res_hop_setup<R, LINK>(a, 1, h, mu, odd[p]);
    res_hop_setup<R, LINK>(a, 0, h, mu, even[p]);
#pragma unroll
    for (int r = 0; r < NR; r++) {
      rv[p][r] = ((const C *)a.basis)[(long)(r < a.nvec ? r : a.nvec - 1) * 3 * Vh + own[p]];
      qv[p][r] = rv[p][r];
    }
  }
  for (int i = threadIdx.x; i < NR * kMaxShifts; i += blockDim.x) {
    const int r = i / kMaxShifts, k = i % kMaxShifts;
    s.z1[r][k] = s.z2[r][k] = 1.0;
    s.flag[r][k] = k < a.nshift;
    s.its[r][k] = 0;
    s.shift[r][k] = r < a.nvec && k < a.nshift ? a.ms[r].shift[k] : 0.0;
  }
  if (threadIdx.x < NR) {
    const int r = threadIdx.x;
    const bool in = r < a.nvec;
    s.diag[r] = in ? a.diag[r] : 0.0;
    s.rho1[r] = in ? a.sh[r].rho1 : 0.0;
    s.rho2[r] = 1.0;
    s.alpha[r] = 1.0;
    s.beta[r] = 0.0;
    s.stop[r] = in ? a.sh[r].stop[1] : 1;
    s.next[r] = s.stop[r];
    s.omega[r] = s.omega_prev[r] = 1.0;
    s.gammag[r] = 0.0;
    s.delta[r] = in ? a.ms[r].delta : 0.0;
    s.res[r] = in ? a.ms[r].res : 0.0;
    s.max_iter[r] = in ? a.ms[r].max_iter : 0;
    s.iter[r] = s.bad[r] = 0;
    s.nact[r] = a.nshift;
    if (r == 0) s.aborted = 0;
  }
  ResLinks<R, LINK> lo, le;  // links of the odd and the even site
  if constexpr (kHeld || kAhead) res_links<R, LINK>(a, odd[0], lo);
  if constexpr (kHeld) res_links<R, LINK>(a, even[0], le);
  __syncthreads();
  for (int k = 1;; k++) {
    bool st[NR];
    bool all = true;
#pragma unroll
    for (int r = 0; r < NR; r++) {
      st[r] = s.stop[r] != 0;
      all &= st[r];
    }
    if (all) break;
    // A: h = D_oe r^(k-1), |h|^2
    double v[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) v[r] = 0.0;
    const C *rin = (const C *)a.basis + (long)(k - 1) * a.stride;
    C *hs = (C *)a.h + (long)(k - 1) * a.stride;
#pragma unroll
    for (int p = 0; p < P; p++) {
      if constexpr (!kHeld && !kAhead) res_links<R, LINK>(a, odd[p], lo);
      if constexpr (kHeld) res_keep(lo);
#pragma unroll
      for (int r0 = 0; r0 < NR; r0 += NB) {
        C o[NB];
        res_hop<R, LINK, NB>(odd[p], lo, rin, Vh, r0, a.nvec, mu, o);
#pragma unroll
        for (int q = 0; q < NB; q++) {
          const int r = r0 + q;
          const C x = cscale(o[q], (R)0.5);
          const bool put = mine[p] && !st[r];
          if (put) {
            res_put(hs + (long)r * 3 * Vh + own[p], x);
            v[r] += (double)x.x * (double)x.x + (double)x.y * (double)x.y;
          }
        }
      }
    }
    res_arrive<NR>(a, s, wg, 2 * k - 2, v);
    if constexpr (kAhead) res_links<R, LINK>(a, even[0], le);
    // while the sums travel: the recurrences of iteration k-1 (bms_step),
    // wave w for systems w, w + nw, ..., a shift per lane
    for (int r = w; r < a.nvec; r += nw) {
      if (s.stop[r]) continue;
      int stop = 0;
      if (k >= 2) {
        const int kk = k - 1;
        const double omp = s.omega[r], gold = s.gammag[r], om = -s.alpha[r], gam = s.beta[r];
        const double rho1 = s.rho1[r], rho2 = s.rho2[r];
        int live = 0;
        if (lane < a.nshift && s.flag[r][lane]) {
          const double z1 = s.z1[r][lane], z2 = s.z2[r][lane];
          const double z3 = (z1 * z2 * omp) / (om * gold * (z1 - z2) + z1 * omp * (1.0 - s.shift[r][lane] * om));
          const double oms = om * z3 / z2;
          const double gas = gam * z3 * oms / (z2 * om);
          if (wg == 0) {
            BmsHist &hh = a.hist[((long)r * a.cap + kk) * a.nshift + lane];
            hh.om = oms;
            hh.z = z3;
            hh.ga = gas;
          }
          live = !(sqrt(rho2 * z2 * z2) < s.res[r]);
          if (!live) {
            s.flag[r][lane] = 0;
            s.its[r][lane] = kk;
          }
          s.z1[r][lane] = z2;
          s.z2[r][lane] = z3;
        }
        const int nact = __popcll(__ballot(live));
        stop = !(sqrt(rho1) > s.res[r] && kk < s.max_iter[r]) || nact == 0 || kk + 2 >= a.cap;
        const bool bad = !isfinite(rho1) || !isfinite(gam) || !isfinite(om);
        if (bad) stop = 1;
        if (lane == 0) {
          s.omega_prev[r] = omp;
          s.omega[r] = om;
          s.gammag[r] = gam;
          s.delta[r] = rho1;
          s.iter[r] = kk;
          s.nact[r] = nact;
          if (bad) s.bad[r] = 1;
        }
      }
      if (lane == 0) s.next[r] = stop;
    }
    if (!res_wait<NR>(a, s, wg, copy, wait, 2 * k - 2)) break;
    if (threadIdx.x < NR) {  // alpha and c of the system (bms_alpha)
      const int r = threadIdx.x;
      double h2 = 0.0;
      for (int q = 0; q < nw; q++) h2 += s.wave[1][q][r];
      const double rho1 = s.rho1[r], b = s.beta[r], ap = s.alpha[r];
      const double mu2 = s.diag[r] * rho1 + h2;
      const double pap = k >= 2 ? mu2 - b * rho1 / ap : mu2;
      const double alpha = rho1 / pap;
      s.coef[0][r] = alpha;
      s.coef[1][r] = k >= 2 && ap != 0.0 ? alpha * b / ap : 0.0;
    }
    __syncthreads();
    // B: r^(k) = r^(k-1) - alpha M^dag M r^(k-1) + c (r^(k-1) - r^(k-2)), |r^(k)|^2
    C *rout = (C *)a.basis + (long)k * a.stride;
    const bool room = k < a.cap;
#pragma unroll
    for (int r = 0; r < NR; r++) v[r] = 0.0;
#pragma unroll
    for (int p = 0; p < P; p++) {
      if constexpr (!kHeld && !kAhead) res_links<R, LINK>(a, even[p], le);
      if constexpr (kHeld) res_keep(le);
#pragma unroll
      for (int r0 = 0; r0 < NR; r0 += NB) {
        C o[NB];
        res_hop<R, LINK, NB>(even[p], le, hs, Vh, r0, a.nvec, mu, o);
#pragma unroll
        for (int q = 0; q < NB; q++) {
          const int r = r0 + q;
          const R d = dg[r], al = (R)s.coef[0][r], c1 = (R)s.coef[1][r];
          C x, rn;
          x.x = fmar(d, rv[p][r].x, (R)-0.5 * o[q].x);
          x.y = fmar(d, rv[p][r].y, (R)-0.5 * o[q].y);
          rn.x = fmar(c1, rv[p][r].x - qv[p][r].x, fmar(-al, x.x, rv[p][r].x));
          rn.y = fmar(c1, rv[p][r].y - qv[p][r].y, fmar(-al, x.y, rv[p][r].y));
          const bool put = mine[p] && !st[r];
          if (put) {
            if (room) res_put(rout + (long)r * 3 * Vh + own[p], rn);
            v[r] += (double)rn.x * (double)rn.x + (double)rn.y * (double)rn.y;
          }
          qv[p][r] = rv[p][r];
          rv[p][r] = rn;
        }
      }
    }
    res_arrive<NR>(a, s, wg, 2 * k - 1, v);
    if constexpr (kAhead) res_links<R, LINK>(a, odd[0], lo);
    if (!res_wait<NR>(a, s, wg, copy, wait, 2 * k - 1)) break;
    if (threadIdx.x < NR) {
      const int r = threadIdx.x;
      if (!s.stop[r]) {
        double rho = 0.0;
        for (int q = 0; q < nw; q++) rho += s.wave[1][q][r];
        s.rho2[r] = s.rho1[r];
        s.rho1[r] = rho;
        s.beta[r] = rho / s.rho2[r];
        s.alpha[r] = s.coef[0][r];
        s.stop[r] = s.next[r];
      }
    }
    __syncthreads();
  }
  // the systems' final state, by the first workgroup
  if (wg != 0) return;
  if (s.aborted) {
    if (threadIdx.x == 0) a.ms[0].nonfinite = kResAborted;
    return;
  }
  for (int i = threadIdx.x; i < a.nvec * kMaxShifts; i += blockDim.x) {
    const int r = i / kMaxShifts, k = i % kMaxShifts;
    if (k >= a.nshift) continue;
    MsState &m = a.ms[r];
    m.z1[k] = s.z1[r][k];
    m.z2[k] = s.z2[r][k];
    m.flag[k] = s.flag[r][k];
    m.its[k] = s.its[r][k];
  }
  if ((int)threadIdx.x < a.nvec) {
    const int r = threadIdx.x;
    MsState &m = a.ms[r];
    m.omega = s.omega[r];
    m.omega_prev = s.omega_prev[r];
    m.gammag = s.gammag[r];
    m.delta = s.delta[r];
    m.iter = s.iter[r];
    m.nact = s.nact[r];
    m.nonfinite = s.bad[r];
    m.stop = m.done = 1;
  }
}

// The grid is the concatenation of the members' grids, each a multiple of 8
// so that each XCD (workgroups are dealt to the 8 XCDs in turn) has a
// contiguous part of the sites; every member meets on its own.
struct ResGroup {
  ResArgs a[kResMaxMembers];
  unsigned start[kResMaxMembers + 1];
  int n;
  long long wait;  // bound of a wait, ticks of the 100 MHz wall clock
};
static_assert(sizeof(ResGroup) <= 4000, "kernel arguments");

// Waves per SIMD the kernel is compiled for: FP32 with one system, the form
// that several lattices share, keeps two workgroups of 512 lanes per CU (with
// two sites per lane it spills 15 of its 128 registers).
template <typename R, int NR>
constexpr int res_waves() {
  return sizeof(R) == 4 && NR == 1 ? 4 : 2;
}

// P: the most sites per lane of any member
template <typename R, int LINK, int NR, int P>
__global__ __launch_bounds__(64 * kResMaxWaves) __attribute__((amdgpu_waves_per_eu(res_waves<R, NR>()))) void k_bms_resident(ResGroup g) {
  int l = 0;
  while (l + 1 < g.n && blockIdx.x >= g.start[l + 1]) l++;
  const unsigned b = blockIdx.x - g.start[l], n = g.start[l + 1] - g.start[l];
  const int wg = (int)((b & 7u) * (n >> 3) + (b >> 3));
  const ResArgs &a = g.a[l];
  if (wg >= a.nwg) return;
  if constexpr (P == 1) {
    res_body<R, LINK, NR, 1>(a, wg, (int)(b & 7u), g.wait);
  } else {
    if (a.sites == 1) res_body<R, LINK, NR, 1>(a, wg, (int)(b & 7u), g.wait);
    else res_body<R, LINK, NR, 2>(a, wg, (int)(b & 7u), g.wait);
  }
}

// ---- power iterations of a small lattice: n of them per launch on the FP64
// 12-real links, p <- (pa p + pb hop(hop(p)/2)) / |p|, meeting twice per
// iteration as the solver does (the first time without a sum).  p of
// iteration i is in slot (base + i) mod (n + 1) of r.basis, h in slot i of
// r.h, so no slot is read before it is written in a launch.  norms[0] is
// |p|^2 at the start, norms[i] that of iteration i, norms[n+1] the
// iterations run (-1: the grid gave up), norms[n+2] whether the last met the
// test; the launch ends at the first one whose norm changed by at most tol
// relatively.
struct PowArgs {
  ResArgs r;
  double pa, pb, tol;
  double *norms;
  int n, base;
  long long wait;
};

template <int P>
__global__ __launch_bounds__(64 * kResMaxWaves) __attribute__((amdgpu_waves_per_eu(2))) void k_pow_resident(PowArgs q) {
  using C = double2;
  constexpr int LINK = LINK_D12;
  const ResArgs &a = q.r;
  __shared__ ResShared<1> s;
  const int copy = (int)(blockIdx.x & 7u);
  const int wg = (int)((blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3));
  if (wg >= a.nwg) return;
  const long Vh = a.L.Vh;
  const int mu = threadIdx.x & 3, nw = blockDim.x >> 6, spw = blockDim.x >> 2;
  bool mine[P];
  unsigned own[P];
  ResHop<double> odd[P], even[P];
  C pv[P];
  C *ring = (C *)a.basis;
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int site = (wg * P + p) * spw + (int)(threadIdx.x >> 2);
    const bool valid = site < (int)Vh;
    const int h = valid ? site : (int)Vh - 1;
    mine[p] = valid && mu < 3;
    own[p] = (unsigned)((mu < 3 ? mu : 2) * Vh + h);
    res_hop_setup<double, LINK>(a, 1, h, mu, odd[p]);
    res_hop_setup<double, LINK>(a, 0, h, mu, even[p]);
    pv[p] = ring[(long)q.base * a.stride + own[p]];
  }
  if (threadIdx.x == 0) s.aborted = 0;
  ResLinks<double, LINK> lo, le;
  if constexpr (P == 1) {
    res_links<double, LINK>(a, odd[0], lo);
    res_links<double, LINK>(a, even[0], le);
  }
  __syncthreads();
  double n2 = q.norms[0], prev = sqrt(n2);
  int i = 0;
  bool met = false;
  for (; i < q.n && !met; i++) {
    const C *in = ring + (long)((q.base + i) % (q.n + 1)) * a.stride;
    C *out = ring + (long)((q.base + i + 1) % (q.n + 1)) * a.stride, *hs = (C *)a.h + (long)i * a.stride;
    double v[1] = {0.0};
#pragma unroll
    for (int p = 0; p < P; p++) {
      if constexpr (P == 1) res_keep(lo);
      else res_links<double, LINK>(a, odd[p], lo);
      C o[1];
      res_hop<double, LINK, 1>(odd[p], lo, in, Vh, 0, 1, mu, o);
      if (mine[p]) res_put(hs + own[p], cscale(o[0], 0.5));
    }
    res_arrive<1>(a, s, wg, 2 * i, v);
    if (!res_wait<1>(a, s, wg, copy, q.wait, 2 * i)) break;
    const double sc = 1.0 / sqrt(n2), pa = q.pa * sc, pb = q.pb * sc;
#pragma unroll
    for (int p = 0; p < P; p++) {
      if constexpr (P == 1) res_keep(le);
      else res_links<double, LINK>(a, even[p], le);
      C o[1];
      res_hop<double, LINK, 1>(even[p], le, hs, Vh, 0, 1, mu, o);
      pv[p] = make_double2(fmar(pa, pv[p].x, pb * o[0].x), fmar(pa, pv[p].y, pb * o[0].y));
      if (mine[p]) {
        res_put(out + own[p], pv[p]);
        v[0] += pv[p].x * pv[p].x + pv[p].y * pv[p].y;
      }
    }
    res_arrive<1>(a, s, wg, 2 * i + 1, v);
    if (!res_wait<1>(a, s, wg, copy, q.wait, 2 * i + 1)) break;
    n2 = 0.0;
    for (int k = 0; k < nw; k++) n2 += s.wave[1][k][0];
    if (wg == 0 && threadIdx.x == 0) q.norms[i + 1] = n2;
    const double norm = sqrt(n2);
    met = !(fabs(prev - norm) / norm > q.tol);
    prev = norm;
  }
  if (wg == 0 && threadIdx.x == 0) {
    q.norms[q.n + 1] = s.aborted ? -1.0 : (double)i;
    q.norms[q.n + 2] = met ? 1.0 : 0.0;
  }
}

}  // namespace rhmc
